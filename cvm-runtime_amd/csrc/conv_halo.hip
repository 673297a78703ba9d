// 3 x 3 convolution, stride 1, padding 1, over 64 channels of a pixel-blocked tensor, int8 out, with or without the 2 x 2
// max_pool2d behind it: the filter and the input pixels under a patch of 512 output pixels lie in LDS.
//
// K is short (18 chunks of 32 bytes), so that a wavefront that streams its operands from memory waits for most of them: each input
// byte is asked for nine times, through an L1 that holds less than the rows under the workgroups of a compute unit, and the filter by every
// wavefront.  Here a workgroup requests each byte of a patch once, memory -> LDS, a border of one pixel included, and the filter
// once for all its patches; the K loop reads LDS with offsets known when it is compiled.  Two workgroups share a compute unit: one fetches or stores
// while the other multiplies.
// In LDS the 16 bytes that a lane feeds to a product are a granule, granules of the same channels lie pixel by pixel: the 32 pixels
// of a block are 512 contiguous bytes.  With the pool a block is one corner of 32 windows, and the columns are sorted into
// even and odd ones for that.
// Measured (us between event pairs): against k_conv_wave 64 -> 64 at 16 x 224 x 224 with the pool 46 -> 30, without 51 -> 33, at 50 x 56 x 56 16.6 -> 13; against
// k_conv_big 64 -> 128 at 16 x 112 x 112 29 -> 22 (more channels: conv_halo_blocks).
// Bound by the requests: a patch takes a workgroup 700 clocks of waiting, 5 400 of products (4 608 at the rate of the matrix pipe), 3 400 to 3 900 in
// which its wavefronts are held until their requests are taken, and 1 400 (pool) to 3 500 of requantisation and stores.  No difference: operands requested
// a step ahead or left to the compiler; slower: a workgroup a patch, each with a filter of its own (36 instead of 30); half of the next patch's requests in
// the middle of the products (32).
// The two layers at the head of a VGG are one launch (STEM): the pixels under a patch, a fifth more than are asked for, are computed from the image by the
// first layer's products where they would be fetched, and the largest tensor of the network is neither written nor read:
// 16 x 224 x 224 with the pool 21 + 28 -> 36 us (trace; other sizes: halo_stem_width).
#include <algorithm>

#include "conv_mfma.h"
#include "requant.h"

namespace cvmhip {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int HALO_CHUNKS = 18, HALO_FILTER = 2 * HALO_CHUNKS * 1024, HALO_PIXELS = 512;

alignas(16) __device__ const int g_halo_zero[4] = {0, 0, 0, 0};

struct HaloGeom {
  const int8_t* x;
  const int8_t* wf;
  int8_t* out;
  const int32_t* bias;
  int H, W, OC, tile_bytes;            // tile_bytes: from 32 filter rows to the next 32
  int lo, hi, shift;
  FastDiv div_oc, div_x, div_y;        // channel groups, patches of a row, rows of patches
  int ocs, across, down, patches;
  // STEM: the convolution over a few channels in front of it (row-window form, conv_mfma.h: StemGeom), whose result is the input
  const int8_t* stem_wf;
  const int32_t* stem_bias;
  int hp, wp, stem_lo, stem_hi, stem_shift;
};

__device__ __forceinline__ void halo_request(const void* from, uint32_t lds_at) {
  // (M0 is written for the instruction behind it: a wait state.  The compiler does not count these requests: stores_done_barrier waits)
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(from), "s"(lds_at) : "memory");
}

// shift sixteen results of a lane to int8 (results are int8 whatever they come from: the saturation never acts)
__device__ __forceinline__ v4i halo_pack(const int (&v)[16], int shift) {
  uint32_t d[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) d[q] = shift_to_bytes(v[q * 4], v[q * 4 + 1], v[q * 4 + 2], v[q * 4 + 3], shift);
  return sixteen_channels(d);
}

// 16 sums of a lane as they start, from 32 biases in LDS: element e is channel (e / 4) * 8 + lgrp * 4 + e % 4
__device__ __forceinline__ v16i halo_first(const int* bias, int lgrp) {
  v16i first;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const v4i v = *reinterpret_cast<const v4i*>(bias + q * 8 + lgrp * 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) first[q * 4 + e] = v[e];
  }
  return first;
}

template <bool POOL, int PW, bool STEM>
__global__ void __launch_bounds__(256, 2) k_conv_halo(const HaloGeom a) {
  constexpr int PH = HALO_PIXELS / PW, ROW = PW + 2, PLANE = (PH + 2) * ROW, HALF = ROW / 2;
  constexpr int REQUESTS = (4 * PLANE + 63) / 64;
  __shared__ __attribute__((aligned(16))) int8_t smem[HALO_FILTER + REQUESTS * 1024];
  __shared__ __attribute__((aligned(16))) int s_bias[STEM ? 128 : 64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 31, lgrp = lane >> 5;
  // A workgroup keeps the filter of its channels and takes patches in turn; an eighth of the patches to each XCD, where neighbours share
  // the pixels between them in one L2.
  int slot = blockIdx.x, slots = gridDim.x, begin = 0, end = a.patches;
  if (gridDim.x % (8 * a.ocs) == 0) {
    const int xcd = slot & 7, per = a.patches >> 3, extra = a.patches & 7;
    slot >>= 3;
    slots >>= 3;
    begin = xcd * per + (xcd < extra ? xcd : extra);
    end = begin + per + (xcd < extra ? 1 : 0);
  }
  const int first_patch = (int)fastdiv((unsigned)slot, a.div_oc), oc0 = (slot - first_patch * a.ocs) * 64, stride = (int)fastdiv((unsigned)slots, a.div_oc);
  int patch = begin + first_patch;
  if (patch >= end) return;
  const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) int8_t*)smem;

  const int8_t* filter = a.wf + (int64_t)(oc0 >> 5) * a.tile_bytes + lane * 16;
#pragma unroll
  for (int k = 0; k < 2 * HALO_CHUNKS / 4; ++k) {
    const int c = wave + 4 * k;
    halo_request(filter + (c >= HALO_CHUNKS ? a.tile_bytes + (c - HALO_CHUNKS) * 1024 : c * 1024), lds + (uint32_t)c * 1024u);
  }
  int n, x0, y0;
  auto corner_of = [&](int which) __attribute__((always_inline)) {
    const int line = (int)fastdiv((unsigned)which, a.div_x);
    n = (int)fastdiv((unsigned)line, a.div_y);
    x0 = (which - line * a.across) * PW;
    y0 = (line - n * a.down) * PH;
  };
  // the places of a patch's granules, the same for all patches: row, column, granule of the pixel
  constexpr int MINE = (REQUESTS + 3) / 4;
  int place[MINE];
#pragma unroll
  for (int k = 0; k < MINE; ++k) {
    const int t = (wave + 4 * k) * 64 + lane, g = t / PLANE, q = t - g * PLANE, r = q / ROW, m = q - r * ROW;
    place[k] = g >= 4 ? -1 : r | (POOL ? (m >= HALF ? 2 * (m - HALF) + 1 : 2 * m) : m) << 8 | g << 16;
  }
  auto fetch = [&]() __attribute__((always_inline)) {
    const int corner = (n * a.H + y0 - 1) * a.W + x0 - 1;
#pragma unroll
    for (int k = 0; k < MINE; ++k) {
      if (wave + 4 * k < REQUESTS) {
        const int r = place[k] & 255, c = place[k] >> 8 & 255, g = place[k] >> 16;
        const bool ok = g >= 0 && (unsigned)(y0 - 1 + r) < (unsigned)a.H && (unsigned)(x0 - 1 + c) < (unsigned)a.W;
        const int p = corner + r * a.W + c;
        const uint64_t inside = (uint64_t)(uintptr_t)a.x + (uint32_t)((p >> 5) * 2048 + g * 512 + (p & 31) * 16), outside = (uint64_t)(uintptr_t)g_halo_zero;
        halo_request(reinterpret_cast<const void*>(ok ? inside : outside), lds + HALO_FILTER + (uint32_t)(wave + 4 * k) * 1024u);
      }
    }
  };
  // STEM: the patch's pixels are computed, a block of 32 places after the other to the wavefronts.
  constexpr int STEM_BLOCKS = (PLANE + 127) / 128;
  v4i window[STEM ? STEM_BLOCKS : 1][2], stem_f[2][2];
  int column;   // of this lane, out of the compiler's sight: what it could work out once for all patches would cost registers that the products need
  auto stem_pixel = [&](int k, int& y, int& x) __attribute__((always_inline)) {
    const int q = (wave + 4 * k) * 32 + column, r = q / ROW, m = q - r * ROW;
    y = y0 - 1 + r;
    x = x0 - 1 + (POOL ? (m >= HALF ? 2 * (m - HALF) + 1 : 2 * m) : m);
    return q < PLANE && y >= 0 && y < a.H && x >= 0 && x < a.W;
  };
  auto stem_request = [&]() __attribute__((always_inline)) {
    typedef int v4w __attribute__((ext_vector_type(4), aligned(4)));
    column = lrow;
    asm volatile("" : "+v"(column));
    const int8_t* filter_at = a.stem_wf + column * 16 + lgrp * 512;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int c = 0; c < 2; ++c) stem_f[i][c] = *reinterpret_cast<const v4i*>(filter_at + (i * 3 + c) * 1024);
#pragma unroll
    for (int k = 0; k < STEM_BLOCKS; ++k) {
      int y, x;
      const bool ok = stem_pixel(k, y, x);
      const int at = ok ? ((n * a.hp + y) * a.wp + x) * 4 : 0;   // the first of three rows of 16 bytes
      window[k][0] = *reinterpret_cast<const v4w*>(a.x + (at + lgrp * a.wp * 4));
      window[k][1] = *reinterpret_cast<const v4w*>(a.x + (at + 2 * a.wp * 4));   // (times a filter of zeros in the upper half)
    }
  };
  auto stem_compute = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < STEM_BLOCKS; ++k) {
      int y, x;
      const bool ok = stem_pixel(k, y, x);
      const int q = (wave + 4 * k) * 32 + column;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        v16i sum = halo_first(s_bias + 64 + i * 32, lgrp);
#pragma unroll
        for (int c = 0; c < 2; ++c) sum = __builtin_amdgcn_mfma_i32_32x32x32_i8(stem_f[i][c], window[k][c], sum, 0, 0, 0);
        asm volatile(WAIT_16_PASSES : "+v"(sum));
        int v[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = clamp_uniform(sum[e], a.stem_lo, a.stem_hi);
        const v4i w = halo_pack(v, a.stem_shift);
        if (q < PLANE) *reinterpret_cast<v4i*>(smem + HALO_FILTER + ((i * 2 + lgrp) * PLANE + q) * 16) = ok ? w : v4i{0, 0, 0, 0};
      }
    }
  };
  corner_of(patch);
  if constexpr (STEM) stem_request();
  else fetch();
  if (tid < 64) {
    s_bias[tid] = a.bias ? a.bias[oc0 + tid] : 0;
    if (STEM) s_bias[64 + tid] = a.stem_bias ? a.stem_bias[tid] : 0;
  }
  if (STEM) __syncthreads();
  v16i acc[2][4];
  // this lane's pixel of block 0 at the window's first tap
  const int wy = PW == 64 ? wave : wave * 2 + (lrow >> 4), wx = PW == 64 ? lrow : lrow & 15;   // POOL: its window
  const int origin = POOL ? 2 * wy * ROW + wx : wave * (PW == 32 ? 4 : 2) * ROW + lrow;
  const int8_t* px = smem + HALO_FILTER + (origin + lgrp * PLANE) * 16;
  const int8_t* fl = smem + lane * 16;
  // K by column of the window and half of the channels, and in these by row: the operand of a row of blocks serves three products, the rows below it
  // included.  A step requests what the next one needs and multiplies what the step before requested.
  constexpr int COLS = POOL || PW == 64 ? 2 : 1, ROWS = 4 / COLS;   // blocks of a wavefront
  v4i f[2][2], b[2][ROWS + 2][COLS];
  auto request = [&](const int t) __attribute__((always_inline)) {
    const int s = t / 6, half = t / 3 % 2, r = t % 3;
#pragma unroll
    for (int i = 0; i < 2; ++i) f[t & 1][i] = *reinterpret_cast<const v4i*>(fl + (i * HALO_CHUNKS + (r * 3 + s) * 2 + half) * 1024);
#pragma unroll
    for (int y = r == 0 ? 0 : ROWS + r - 1; y < ROWS + r; ++y)
#pragma unroll
      for (int x = 0; x < COLS; ++x) {
        const int at = y * ROW + (POOL ? ((x + s) & 1) * HALF + ((x + s) >> 1) : x * 32 + s);
        b[t / 3 & 1][y][x] = *reinterpret_cast<const v4i*>(px + (half * 2 * PLANE + at) * 16);
      }
  };
  for (;;) {
    if constexpr (STEM) stem_compute();
    stores_done_barrier();   // the requests have landed
    request(0);
    const v16i first[2] = {halo_first(s_bias, lgrp), halo_first(s_bias + 32, lgrp)};
#pragma unroll
    for (int t = 0; t < HALO_CHUNKS; ++t) {
      if (t + 1 < HALO_CHUNKS) request(t + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f[t & 1][i], b[t / 3 & 1][j / COLS + t % 3][j % COLS], t == 0 ? first[i] : acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }

    const int now_n = n, now_x = x0, now_y = y0;
    patch += stride;
    const bool more = patch < end;
    __syncthreads();   // the patch has been read
    if (more) {
      corner_of(patch);
      if constexpr (!STEM) fetch();
    }
    asm volatile(WAIT_16_PASSES : "+v"(acc[0][0]), "+v"(acc[0][1]), "+v"(acc[0][2]), "+v"(acc[0][3]), "+v"(acc[1][0]), "+v"(acc[1][1]), "+v"(acc[1][2]),
                 "+v"(acc[1][3]));
    const int OW = POOL ? a.W >> 1 : a.W, OH = POOL ? a.H >> 1 : a.H;
    const int cblocks = a.OC >> 5;
#pragma unroll
    for (int j = 0; j < (POOL ? 1 : 4); ++j) {
      const int y = POOL ? (now_y >> 1) + wy : PW == 32 ? now_y + wave * 4 + j : now_y + wave * 2 + (j >> 1);
      const int x = POOL ? (now_x >> 1) + wx : PW == 32 ? now_x + lrow : now_x + (j & 1) * 32 + lrow;
      const int p = (now_n * OH + y) * OW + x;
      const bool ok = y < OH && x < OW;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        int v[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          int m = acc[i][j][e];
          if (POOL) m = max(max(m, acc[i][1][e]), max(acc[i][2][e], acc[i][3][e]));
          v[e] = clamp_uniform(m, a.lo, a.hi);
        }
        const v4i w = halo_pack(v, a.shift);
        if (ok) {
          const int64_t at = ((int64_t)(p >> 5) * cblocks + (oc0 >> 5) + i) * 1024 + lgrp * 512 + (p & 31) * 16;
          __builtin_nontemporal_store(w, reinterpret_cast<v4i*>(a.out + at));
        }
      }
    }
    if (!more) break;
    if constexpr (STEM) stem_request();   // (in front of the requantisation the registers do not suffice)
  }
}

// the patch that covers the image with fewer pixels outside it
static int halo_width(int h, int w) {
  const int64_t a = (int64_t)((w + 31) / 32) * ((h + 15) / 16), b = (int64_t)((w + 63) / 64) * ((h + 7) / 8);
  return a <= b ? 32 : 64;
}
static int64_t halo_patches(const ConvGeom& g, int width) {
  return (int64_t)g.N * ((g.W + width - 1) / width) * ((g.H + HALO_PIXELS / width - 1) / (HALO_PIXELS / width));
}
static int64_t halo_patches(const ConvGeom& g) { return halo_patches(g, halo_width(g.H, g.W)); }

// one clamp and one shift to int8
static bool halo_chain(const DevChain& c, int* lo, int* hi, int* shift) { return clamp_shift_of(c, lo, hi, shift) && clamp_shift_narrow(*lo, *hi, *shift); }

// Is it such a layer?  (g and ep as conv_prepare leaves them)
static bool halo_layer(const ConvGeom& g, const Epilogue& ep) {
  if (g.dw || g.row_bytes || g.Cp != 64 || g.OC % 64 != 0 || g.KH != 3 || g.KW != 3 || g.SH != 1 || g.SW != 1 || g.PH != 1 || g.PW != 1 || g.DH != 1 ||
      g.DW != 1 || ep.out_mode != OUT_I8_ACT || ep.out_cp != g.OC || ep.residual || ep.split)
    return false;
  int lo, hi, shift;
  return (int64_t)g.N * g.H * g.W * 64 <= INT32_MAX && halo_patches(g) * (g.OC / 64) <= INT32_MAX && halo_chain(ep.chain, &lo, &hi, &shift);
}
// From 150 workgroups on (us here / k_conv_wave, 64 channels at 56 x 56: 112 workgroups 9.4 / 9.0, 140 9.9 / 9.6, 168 10.2 / 11.4, 224 10.8 / 13.4), and
// where the patches have at most half as many pixels again as the image (64 x 100 x 75, 1.43 times: 26.7 / 29.9; 128 x 33 x 48, 1.62: 16.9 / 15.8).
static bool halo_fills(const ConvGeom& g) {
  const int64_t patches = halo_patches(g);
  return patches * (g.OC / 64) >= 150 && patches * HALO_PIXELS * 2 <= (int64_t)g.N * g.H * g.W * 3;
}

// Without the pool also only past the 512 tiles of 64 channels x 128 pixels up to which k_conv_wave splits K over its wavefronts and is through in one
// round.  Layers of 150 to 200 workgroups here (their patches 1.14 to 1.49 times the image), us here / there: with up to 512 such tiles 9.3-9.8 / 8.8-9.3
// whatever the channels (64 to 384), with more 9.5-10.2 / 10.6-12.9; with the pool 8.3-8.5 / 8.9-10.5 on the near side of the line as well.
// 192 channels are a tile and a half of k_conv_big, which would have such a layer from 160 tiles on: 9.4-9.7 / 12.4-12.6 between the two lines.
// More channels (before it k_conv_big): 8 x 56 x 56 to 192 10.0 / 12.9, 16 x 28 x 28 to 512 10.3 / 13.2, 32 x 56 x 56 to 320 28.8 / 39.0 (with the pool
// 22.6 / 30.7), 16 x 112 x 112 to 256 37.2 / 50.4; the least, 16 x 75 x 75 to 512, 40.5 / 44.0.
int64_t conv_halo_blocks(const ConvGeom& g, const Epilogue& ep) {
  if (!halo_layer(g, ep) || !halo_fills(g)) return 0;
  const int64_t pixels = (int64_t)g.N * g.H * g.W;
  const bool one_round = (pixels + 127) / 128 * (g.OC / 64) <= 512, large = g.OC > 64 && (pixels + 255) / 256 * ((g.OC + 127) / 128) >= 160;
  if (!ep.pool && one_round && !large) return 0;
  return halo_patches(g) * (g.OC / 64);
}

static void halo_geom(HaloGeom* a, const int8_t* wp, void* out, const ConvGeom& g, const Epilogue& ep, int width) {
  a->wf = wp;
  a->out = reinterpret_cast<int8_t*>(out);
  a->bias = ep.bias;
  a->H = g.H; a->W = g.W; a->OC = g.OC;
  a->tile_bytes = (HALO_CHUNKS + 1) * 1024;
  halo_chain(ep.chain, &a->lo, &a->hi, &a->shift);
  a->ocs = g.OC / 64;
  a->patches = (int)halo_patches(g, width);
  a->across = (g.W + width - 1) / width;
  a->down = (g.H + HALO_PIXELS / width - 1) / (HALO_PIXELS / width);
  a->div_oc = make_fastdiv((uint32_t)a->ocs);
  a->div_x = make_fastdiv((uint32_t)a->across);
  a->div_y = make_fastdiv((uint32_t)a->down);
}

template <bool STEM>
static int halo_launch(const HaloGeom& a, bool pool, int width, hipStream_t s) {
  const int at_once = std::max(1, 512 / a.ocs);   // patches: two workgroups a compute unit
  const unsigned grid = (unsigned)(a.ocs * std::min(a.patches, at_once));
  if (pool && width == 32) k_conv_halo<true, 32, STEM><<<grid, 256, 0, s>>>(a);
  else if (pool) k_conv_halo<true, 64, STEM><<<grid, 256, 0, s>>>(a);
  else if (width == 32) k_conv_halo<false, 32, STEM><<<grid, 256, 0, s>>>(a);
  else k_conv_halo<false, 64, STEM><<<grid, 256, 0, s>>>(a);
  return check_launch("conv_halo");
}

int conv_halo(const int8_t* xp, const int8_t* wp, void* out, const ConvGeom& g, const Epilogue& ep, hipStream_t s) {
  const int width = halo_width(g.H, g.W);
  HaloGeom a = {};
  a.x = xp;
  halo_geom(&a, wp, out, g, ep, width);
  return halo_launch<false>(a, ep.pool != 0, width, s);
}

// The first two layers of a VGG in one launch: where halo_fills.  206 cases of 150 to 1 568 patches, up to 1.49 times the image, with the pool and without it, against
// the faster of the two launches with k_conv_halo and with k_conv_wave for the second layer: 0.95 to 1.45 times as fast, 1.19 in the middle (us here / there:
// 2 x 224 x 224 12.4 / 16.3, 4 x 224 x 224 17.2 / 20.3, 2 x 300 x 300 16.8 / 23.6, 43 x 46 x 46 15.4 / 16.0, 58 x 38 x 90 22.0 / 23.4, 300 x 24 x 30 22.4 / 23.9).
// Patches of 64 x 8 need six blocks of the first layer for each wavefront instead of five, 1.14 times the time: 35 x 36 x 180 25.7 / 24.8, where 32 x 16
// takes 22.6.  Time goes by rounds of 256 patches, one to a compute unit, so the wide ones stay where they save a round: 14 x 66 x 128 14.4 instead of 15.5,
// 133 x 24 x 44 18.1 instead of 20.8.  (Slower than two launches: 233 x 24 x 44 and the like, 700 wide patches of 1.45 times the image, 26.2 / 25.2.)
static int halo_stem_width(const ConvGeom& g) {
  const int64_t narrow = (halo_patches(g, 32) + 255) / 256, wide = (halo_patches(g, 64) + 255) / 256;
  return wide * 8 < narrow * 7 ? 64 : 32;
}
static bool halo_stem_prepare(const cvmhip_chain* stem_chain, const cvmhip_chain* chain, int n, int c, int h, int w, int pool, ConvGeom* g, Epilogue* ep,
                              HaloGeom* a, StemGeom* sg) {
  if (n < 1 || c < 1 || c > 4 || h < 1 || w < 1 || (pool && (h % 2 || w % 2)) || cvmhip_stem_input_bytes(n, h, w, 3, 3, 1, 1, 1, 1) == 0) return false;
  *sg = stem_geom(n, h, w, 3, 3, 1, 1, 1, 1);
  if (sg->bytes > INT32_MAX || sg->row_bytes != 16) return false;
  DevChain first;
  if (!make_chain(stem_chain, &first) || !halo_chain(first, &a->stem_lo, &a->stem_hi, &a->stem_shift) || !make_chain(chain, &ep->chain)) return false;
  g->N = n; g->H = g->OH = h; g->W = g->OW = w; g->Cp = g->OC = 64;
  g->KH = g->KW = 3; g->SH = g->SW = g->PH = g->PW = g->DH = g->DW = 1;
  ep->out_mode = OUT_I8_ACT;
  ep->out_cp = 64;
  ep->pool = pool;
  return halo_layer(*g, *ep) && halo_fills(*g) && halo_patches(*g, halo_stem_width(*g)) <= INT32_MAX;
}

}  // namespace cvmhip

using namespace cvmhip;

extern "C" {

int cvmhip_conv2d_stem_conv_i8_eligible(const cvmhip_chain* stem_chain, const cvmhip_chain* chain, int n, int c, int h, int w, int pool) {
  ConvGeom g = {};
  Epilogue ep = {};
  HaloGeom a = {};
  StemGeom sg;
  return stem_chain && chain && halo_stem_prepare(stem_chain, chain, n, c, h, w, pool, &g, &ep, &a, &sg) ? 1 : 0;
}

int cvmhip_conv2d_stem_conv_i8(const void* xs, const void* stem_wp, const int32_t* stem_bias, const cvmhip_chain* stem_chain, const void* wp, const int32_t* bias,
                               const cvmhip_chain* chain, void* out, int n, int c, int h, int w, int pool, void* stream) {
  ConvGeom g = {};
  Epilogue ep = {};
  HaloGeom a = {};
  StemGeom sg;
  if (!xs || !stem_wp || !stem_chain || !wp || !chain || !out || (((uintptr_t)xs | (uintptr_t)stem_wp | (uintptr_t)wp | (uintptr_t)out) & 15) ||
      !halo_stem_prepare(stem_chain, chain, n, c, h, w, pool, &g, &ep, &a, &sg))
    return arg_error("conv2d_stem_conv_i8: not eligible");
  ep.bias = bias;
  const int width = halo_stem_width(g);
  a.x = reinterpret_cast<const int8_t*>(xs);
  halo_geom(&a, reinterpret_cast<const int8_t*>(wp), out, g, ep, width);
  a.stem_wf = reinterpret_cast<const int8_t*>(stem_wp);
  a.stem_bias = stem_bias;
  a.hp = sg.hp; a.wp = sg.wp;
  char desc[128] = "";
  if (kernel_timing_enabled()) snprintf(desc, sizeof(desc), "3x3/1 %d->64 and 3x3/1 64->64 in %dx%dx%d%s, patches of %d x %d", c, n, h, w, pool ? " +pool" : "", width,
                                        HALO_PIXELS / width);
  KernelTimer timer("k_conv_halo", 2.0 * n * h * w * 64 * 9 * (64.0 + c), as_stream(stream),
                    4.0 * n * sg.hp * sg.wp + 64.0 * 9 * (64 + c) + (double)n * h * w * 64 / (pool ? 4 : 1), desc);
  return halo_launch<true>(a, pool != 0, width, as_stream(stream));
}

}  // extern "C"
