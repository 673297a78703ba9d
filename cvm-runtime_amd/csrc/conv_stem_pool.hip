// The head of a ResNet at larger batches: a 7 x 7 convolution with stride 2 over a few channels (row-window form, conv_mfma.h:
// StemGeom), 64 channels out, and max_pool2d with a 3 x 3 window, stride 2 and padding 1 behind it, in one launch.
//
// As two launches the convolution's output is written and read, four times what the pool leaves.  Here a workgroup takes patches of
// 8 x 14 pooled pixels in turn: the 17 x 29 convolution pixels under a patch are 16 blocks of 32 with hardly a lane to spare, their input
// rows lie in LDS, the filter in registers, and the results as int8 in LDS, where the maxima are taken.  The next patch's input is requested
// in front of the products and put to LDS behind them.
// Measured at 224 x 224 (us; convolution and pool as two launches in front of it): batch 16 18.1 -> 10.2, batch 50 43 -> 22; three workgroups a compute unit, bound by
// the chain of each patch (products 1 800 clocks a SIMD, requantisation 1 400, maxima 800, two barriers) and the input's way.
// (k_stem_pool, with smaller patches and every operand from memory, stays for small batches: there are enough workgroups to answer fast.)
#include <algorithm>

#include "conv_mfma.h"
#include "requant.h"

namespace cvmhip {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int HEAD_QH = 8, HEAD_QW = 14, HEAD_CH = 2 * HEAD_QH + 1, HEAD_CW = 2 * HEAD_QW + 1, HEAD_K = 7;
constexpr int HEAD_ROWS = 2 * (HEAD_CH - 1) + HEAD_K, HEAD_GRANULES = (2 * (HEAD_CW - 1) + 8) * 4 / 16 + 1;   // input rows, 16 bytes of a row (one more: see delta)
constexpr int HEAD_PITCH = HEAD_GRANULES * 16, HEAD_LOADS = (HEAD_ROWS * HEAD_GRANULES + 255) / 256;
constexpr int HEAD_PIXELS = 512;
static_assert(HEAD_CH * HEAD_CW <= HEAD_PIXELS, "four blocks a wavefront");

struct HeadGeom {
  const int8_t* xs;
  const int8_t* wf;
  int8_t* out;
  const int32_t* bias;
  int hp, wp, last;              // stored input; byte offset of the last 16 bytes
  int OH, OW, QH, QW;
  int tile_bytes, patches, across, down;
  FastDiv div_x, div_y;
  int plain, lo, hi, shift;      // the chain is one clamp and one shift to int8
  DevChain chain;
};

__global__ void __launch_bounds__(256, 2) k_conv_stem_pool(const HeadGeom a) {
  __shared__ __attribute__((aligned(16))) int8_t s_tile[4 * HEAD_PIXELS * 16];   // [16 channels][convolution pixel of the patch]
  __shared__ __attribute__((aligned(16))) int8_t s_in[HEAD_ROWS * HEAD_PITCH];
  __shared__ __attribute__((aligned(16))) int s_bias[64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 31, lgrp = lane >> 5;
  // an eighth of the patches to each XCD: neighbours share input rows in one L2
  int slot = blockIdx.x, slots = gridDim.x, begin = 0, end = a.patches;
  if (gridDim.x % 8 == 0) {
    const int xcd = slot & 7, per = a.patches >> 3, extra = a.patches & 7;
    slot >>= 3;
    slots >>= 3;
    begin = xcd * per + (xcd < extra ? xcd : extra);
    end = begin + per + (xcd < extra ? 1 : 0);
  }
  int patch = begin + slot;
  if (patch >= end) return;
  if (tid < 64) s_bias[tid] = a.bias ? a.bias[tid] : 0;
  v4i f[2][HEAD_K];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < HEAD_K; ++r) f[i][r] = *reinterpret_cast<const v4i*>(a.wf + i * a.tile_bytes + r * 1024 + lane * 16);
  int ry[4], rx[4];   // this lane's pixel of each of its blocks
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int u = (wave * 4 + j) * 32 + lrow;
    ry[j] = u / HEAD_CW;
    rx[j] = u - ry[j] * HEAD_CW;
    if (ry[j] >= HEAD_CH) ry[j] = HEAD_CH - 1;   // (lanes without a pixel repeat one; nobody reads what they leave)
  }

  int n, cy0, cx0, delta;
  v4i next[HEAD_LOADS];
  // The first column of a patch at the left edge is one that does not exist: its input begins with the row then, and `delta` moves the reads.
  auto request = [&](int which) __attribute__((always_inline)) {
    const int line = (int)fastdiv((unsigned)which, a.div_x);
    n = (int)fastdiv((unsigned)line, a.div_y);
    cy0 = 2 * (line - n * a.down) * HEAD_QH - 1;
    cx0 = 2 * (which - line * a.across) * HEAD_QW - 1;
    const int c0 = cx0 < 0 ? 0 : 2 * cx0;
    delta = 2 * cx0 - c0;
    typedef int v4w __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
    for (int k = 0; k < HEAD_LOADS; ++k) {
      const int t = tid + 256 * k, r = t / HEAD_GRANULES, g = t - r * HEAD_GRANULES;
      int y = 2 * cy0 + r;
      y = y < 0 ? 0 : (y > a.hp - 1 ? a.hp - 1 : y);
      int at = ((n * a.hp + y) * a.wp + c0) * 4 + g * 16;   // (bytes past the row or the tensor belong to pixels that do not exist)
      at = at < a.last ? at : a.last;
      next[k] = *reinterpret_cast<const v4w*>(a.xs + at);
    }
  };
  auto place = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < HEAD_LOADS; ++k) {
      const int t = tid + 256 * k;
      if (t < HEAD_ROWS * HEAD_GRANULES) *reinterpret_cast<v4i*>(s_in + t * 16) = next[k];
    }
  };
  request(patch);
  place();
  for (;;) {
    __syncthreads();   // the input is there, and the tile has been read
    const int now_n = n, now_y = cy0, now_x = cx0, now_delta = delta;
    patch += slots;
    const bool more = patch < end;
    if (more) request(patch);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v16i acc[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const v4i v = *reinterpret_cast<const v4i*>(s_bias + i * 32 + q * 8 + lgrp * 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][q * 4 + e] = v[e];
        }
      int col = (2 * rx[j] + now_delta) * 4 + lgrp * 16;
      col = col < 0 ? 0 : col;   // (the column that does not exist)
      const int8_t* px = s_in + 2 * ry[j] * HEAD_PITCH + col;
#pragma unroll
      for (int r = 0; r < HEAD_K; ++r) {
        const v2i b0 = *reinterpret_cast<const v2i*>(px + r * HEAD_PITCH), b1 = *reinterpret_cast<const v2i*>(px + r * HEAD_PITCH + 8);
        const v4i b = {b0[0], b0[1], b1[0], b1[1]};
#pragma unroll
        for (int i = 0; i < 2; ++i) acc[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f[i][r], b, acc[i], 0, 0, 0);
      }
      asm volatile(WAIT_16_PASSES : "+v"(acc[0]), "+v"(acc[1]));
      const int cy = now_y + ry[j], cx = now_x + rx[j];
      const bool inside = cy >= 0 && cy < a.OH && cx >= 0 && cx < a.OW;
      const int u = (wave * 4 + j) * 32 + lrow;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        uint32_t d[4];
        if (a.plain) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            int v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = clamp_uniform(acc[i][q * 4 + e], a.lo, a.hi);
            d[q] = shift_to_bytes(v[0], v[1], v[2], v[3], a.shift);   // (results are int8 whatever they come from: the saturation never acts)
          }
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            int v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = apply_chain(a.chain, acc[i][q * 4 + e]);
            d[q] = low_bytes(v[0], v[1], v[2], v[3]);
          }
        }
        const int none = (int)0x80808080u;   // outside the convolution's output: less than any value (a window holds at least one)
        const v4i channels = sixteen_channels(d), w = inside ? channels : v4i{none, none, none, none};
        *reinterpret_cast<v4i*>(s_tile + (i * 2 + lgrp) * HEAD_PIXELS * 16 + u * 16) = w;
      }
    }
    __syncthreads();   // the tile is there, and the input has been read
    if (more) place();
    for (int t = tid; t < 4 * HEAD_QH * HEAD_QW; t += 256) {
      const int g = t / (HEAD_QH * HEAD_QW), q = t - g * (HEAD_QH * HEAD_QW), y = q / HEAD_QW, x = q - y * HEAD_QW;
      const int8_t* from = s_tile + (g * HEAD_PIXELS + 2 * y * HEAD_CW + 2 * x) * 16;
      int4 v[9];
#pragma unroll
      for (int dy = 0; dy < 3; ++dy)
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) v[dy * 3 + dx] = *reinterpret_cast<const int4*>(from + (dy * HEAD_CW + dx) * 16);
      const int qy = (now_y + 1) / 2 + y, qx = (now_x + 1) / 2 + x;
      if (qy < a.QH && qx < a.QW) {
        const int4 m = max_pool_reduce<9>(v);
        __builtin_nontemporal_store(v4i{m.x, m.y, m.z, m.w}, reinterpret_cast<v4i*>(a.out + act_offset((int64_t)(now_n * a.QH + qy) * a.QW + qx, g * 16, 64)));
      }
    }
    if (!more) break;
  }
}

static int64_t head_patches(int n, int qh, int qw) { return (int64_t)n * ((qh + HEAD_QH - 1) / HEAD_QH) * ((qw + HEAD_QW - 1) / HEAD_QW); }

// us here / k_stem_pool / two launches.  Up to 512 tiles of 4 x 8 pooled pixels k_stem_pool runs them all at once; it is the faster one while no compute unit has two
// (3 x 224 x 224, 294 tiles, 8.4 / 8.9; 2 x 224 x 224, 196, 8.4 / 7.5; 27 x 64 x 64, 216, 8.3 / 7.6; 256 tiles 8.1 / 7.5), and where the patches, which are larger, come to a
// second one (36 x 100 x 60, 504 tiles and 288 patches, 11.5 / 9.1).  With 257 to 330 tiles the gain depends on the map: 16 x 96 x 96 8.1 / 9.0, 5 x 171 x 171 9.2 / 8.9.
// Past 512 tiles the alternative is two launches, and what counts is how much of the patches lies outside the map: 16 x 224 x 224, nothing, 11.5 / 22.7 / 20.5;
// 50 x 171 x 171, 1.45 times the map, 19.5 / 37.7 / 29.0; 100 x 68 x 116, 2.04, 15.8 / 24.1 / 19.9; 200 x 100 x 60, 2.39, 25.1 / 32.4 / 26.9; 900 x 17 x 60, 2.99, 25.2 / 40.7 /
// 24.4; 640 x 36 x 60, 3.32, 32.5 / 42.1 / 28.7; 800 x 20 x 20, 4.5, 14.9 / 22.0 / 13.7.
bool conv_stem_pool_takes(int n, int oc, int kh, int kw, int sh, int sw, int qh, int qw) {
  if (oc != 64 || kh != HEAD_K || kw <= 4 || kw > 8 || sh != 2 || sw != 2) return false;
  const int64_t patches = head_patches(n, qh, qw), tiles = stem_pool_tiles(n, qh, qw);
  if (tiles <= STEM_POOL_AT_ONCE) return patches >= 80 && tiles > 256 && patches <= 256;
  return (patches * (HEAD_QH * HEAD_QW) <= 3 * (int64_t)n * qh * qw || n > 65535) && patches <= INT32_MAX;   // (k_stem_pool's grid ends at 65 535 images)
}

int conv_stem_pool(const int8_t* xs, const int8_t* wp, const int32_t* bias, const DevChain& chain, int8_t* out, const StemGeom& sg, int n, int oh, int ow, int qh,
                   int qw, hipStream_t s) {
  HeadGeom a = {};
  a.xs = xs;
  a.wf = wp;
  a.out = out;
  a.bias = bias;
  a.hp = sg.hp; a.wp = sg.wp;
  a.last = (int)sg.bytes - 16;
  a.OH = oh; a.OW = ow; a.QH = qh; a.QW = qw;
  a.tile_bytes = (sg.kp / 32 + 1) * 1024;
  a.across = (qw + HEAD_QW - 1) / HEAD_QW;
  a.down = (qh + HEAD_QH - 1) / HEAD_QH;
  a.patches = (int)head_patches(n, qh, qw);
  a.div_x = make_fastdiv((uint32_t)a.across);
  a.div_y = make_fastdiv((uint32_t)a.down);
  a.chain = chain;
  a.plain = clamp_shift_of(chain, &a.lo, &a.hi, &a.shift) && clamp_shift_narrow(a.lo, a.hi, a.shift);
  k_conv_stem_pool<<<(unsigned)std::min(a.patches, 768), 256, 0, s>>>(a);
  return check_launch("conv2d_stem_pool3_i8");
}

}  // namespace cvmhip
