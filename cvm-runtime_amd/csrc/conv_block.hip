// The tail of a ResNet bottleneck and the head of the next one, one launch for three layers:
//   A  3 x 3, padding 1, stride 1 or 2, M -> M channels
//   B  1 x 1, M -> 4 M, the residual added
//   C  1 x 1, 4 M -> M or 2 M (the first layer of the next block)
// with M = 64, 128 or 256; B's result is stored (the next block's residual), A's never leaves the compute unit and C reads B's where it was made.
//
// As launches of their own the three are bound by what surrounds their products: a launch, the first operands' way, a partial last round and a
// tensor of 4 M channels written and fetched again.  Here a workgroup of eight wavefronts computes all channels of all three layers for a tile of
// 16 * NT consecutive output pixels.  The pixels under the 3 x 3 windows, a run of the input's pixels, are fetched into LDS once, and the residual
// to where B's result will lie; A's and B's results stay in LDS, pixel by pixel, as the operand of the layer behind.  The filters are not shared inside a
// workgroup (each wavefront has channels of its own), so they go from memory to registers: a wavefront's fragments of all three layers are one stream,
// requested RING fragments ahead across the layers.
// v_mfma_i32_16x16x64_i8 with the filter as first operand: a lane's four results are four consecutive channels of one pixel, a dword of the operand.
#include <algorithm>
#include <numeric>

#include "conv_mfma.h"
#include "requant.h"

namespace cvmhip {

typedef int v4i __attribute__((ext_vector_type(4)));

alignas(16) __device__ const int g_block_zero[4] = {0, 0, 0, 0};

struct BlockRequant { int lo, hi, shift; };
struct BlockArgs {
  const int8_t *x, *wa, *wb, *wc, *res;   // res: the residual, or what the projection reads that makes it
  const int8_t* ws;
  const int32_t *ba, *bb, *bc, *bs;
  int8_t *out, *next;
  int H, W, S, P, in_pixels;          // input extent, stride of A, output pixels and input pixels of all images
  int patch, tiles;                   // pixels of a tile's run of the input, tiles
  const int8_t* ahead[3];             // filters of a launch behind this one, which the workgroups past the tiles fetch into the L2 of their XCD
  int ahead_kib[3], helpers;          // and how many of those there are for each XCD (0: none)
  FastDiv div_ohw, div_ow, div_patch;
  int OHW, OW;
  BlockRequant qa, qb, qr, qc, qs;    // qb in front of the residual, qr behind it; qs: the projection's
};

// Where things lie in LDS: sixteen zeros for windows that leave the image, biases, A's result, B's result, the run of the input.  Granules of 16 channels
// lie pixel by pixel, channel group after channel group: a quarter of a wavefront requests, reads and writes 16 neighbouring pixels, and these are
// neighbours in memory too.
// KS: 64-byte steps of K of the projection that makes the residual, 0: none
template <int M, int NT, int UC, int KS>
struct BlockLds {
  static constexpr int P = 16 * NT, GROUP = P * 16;   // bytes of a channel group of A's and B's results
  static constexpr int biases = (5 + UC + (KS ? 4 : 0)) * M, bias_requests = (biases * 4 + 1023) / 1024;
  static constexpr int zero = 0, bias = 64, mid = bias + bias_requests * 1024, wide = mid + M / 16 * GROUP, cut = wide + M / 4 * GROUP, patch = cut + KS * 4 * GROUP;
  static int64_t bytes(int64_t patch_pixels) { return patch + (patch_pixels * (M / 16) + 63) / 64 * 1024; }
};

__device__ __forceinline__ void block_request(const void* from, uint32_t lds_at) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(from), "s"(lds_at) : "memory");
}
// all but the last N requests of this wavefront have landed (they do so in order)
template <int N>
__device__ __forceinline__ void block_landed() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N < 63 ? N : 63) : "memory"); }
// LDS written before is read behind it; requests of memory stay in flight
__device__ __forceinline__ void block_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// (the wait is part of the values' way, see WAIT_8_PASSES)
template <int N, int I = 0>
__device__ __forceinline__ void block_settle(v4i (&acc)[N]) {
  if constexpr (N - I >= 8) {
    asm volatile(WAIT_8_PASSES : "+v"(acc[I]), "+v"(acc[I + 1]), "+v"(acc[I + 2]), "+v"(acc[I + 3]), "+v"(acc[I + 4]), "+v"(acc[I + 5]), "+v"(acc[I + 6]), "+v"(acc[I + 7]));
    block_settle<N, I + 8>(acc);
  } else if constexpr (N - I >= 4) {
    asm volatile(WAIT_8_PASSES : "+v"(acc[I]), "+v"(acc[I + 1]), "+v"(acc[I + 2]), "+v"(acc[I + 3]));
    block_settle<N, I + 4>(acc);
  } else if constexpr (N - I >= 2) {
    asm volatile(WAIT_8_PASSES : "+v"(acc[I]), "+v"(acc[I + 1]));
    block_settle<N, I + 2>(acc);
  } else if constexpr (N - I == 1) {
    asm volatile(WAIT_8_PASSES : "+v"(acc[I]));
  }
}

template <int M, int NT, int UC, int KS, int RING, int OCC, bool HELPERS>
__global__ void __launch_bounds__(512, 2 * OCC) k_conv_block(const BlockArgs a) {
  typedef BlockLds<M, NT, UC, KS> L;
  constexpr int CTA = M == 256 ? 2 : 1, PGA = M == 64 ? 2 : 1, NTA = NT / PGA;   // A and C: 16-channel tiles of a wavefront at a time, groups of pixels
  constexpr int KA = M / 64, UB = M / 64, KC = M / 16;                           // 64-byte steps of K: of a tap, of B (units of 32 channels likewise), of C
  constexpr int FA = 9 * KA * CTA, FS = UB * KS * 2, FB = UB * KA * 2, FC = UC * KC * CTA, F = FA + FS + FB + FC;
  constexpr int TILE_A = (9 * M / 32 + 1) * 1024, TILE_B = (M / 32 + 1) * 1024, TILE_C = (M / 8 + 1) * 1024, TILE_S = (KS * 2 + 1) * 1024;   // from 32 filter rows to the next
  static_assert(NT % PGA == 0, "pixels are split between wavefronts by 16");
  extern __shared__ __attribute__((aligned(16))) int8_t block_lds[];
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, kg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) int8_t*)block_lds;
  if (HELPERS && (int)blockIdx.x >= a.tiles) {
    const int first_kib = (((int)blockIdx.x - a.tiles) >> 3) * 8 + wave;
#pragma unroll
    for (int i = 0; i < 3; ++i)
      for (int k = first_kib; k < a.ahead_kib[i]; k += a.helpers * 8) block_request(a.ahead[i] + (int64_t)k * 1024 + lane * 16, lds + (uint32_t)wave * 1024u);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    return;
  }

  // an eighth of the tiles to each XCD, where neighbours share the pixels between them
  int tile;
  {
    const int xcd = blockIdx.x & 7, per = a.tiles >> 3, extra = a.tiles & 7;
    tile = xcd * per + (xcd < extra ? xcd : extra) + ((int)blockIdx.x >> 3);
  }
  const int p0 = tile * L::P;
  auto corner = [&](int p, int& row, int& column, int& n) __attribute__((always_inline)) {   // of a pixel's window, in the input
    n = (int)fastdiv((unsigned)p, a.div_ohw);
    const int rem = p - n * a.OHW, oh = (int)fastdiv((unsigned)rem, a.div_ow);
    row = oh * a.S - 1;
    column = (rem - oh * a.OW) * a.S - 1;
  };
  int first;   // pixel of the input at the start of the run
  {
    int r, c, n;
    corner(p0, r, c, n);
    first = (n * a.H + r) * a.W + c;
  }

  // ---- biases, then the run of the input
#pragma unroll
  for (int k = 0; k < L::bias_requests; k += 8) {
    if (k + wave < L::bias_requests) {
      const int i = ((k + wave) * 64 + lane) * 4;
      const int32_t* b = i < M ? a.ba : i < 5 * M ? a.bb : i < (5 + UC) * M ? a.bc : a.bs;
      const int at = i < M ? i : i < 5 * M ? i - M : i < (5 + UC) * M ? i - 5 * M : i - (5 + UC) * M;
      block_request(b && i < L::biases ? b + at : g_block_zero, lds + L::bias + (uint32_t)(k + wave) * 1024u);
    }
  }
  const int run_requests = (a.patch * (M / 16) + 63) >> 6;
  for (int k = wave; k < run_requests; k += 8) {
    const int t = k * 64 + lane;
    int g = (int)fastdiv((unsigned)t, a.div_patch), p = first + t - g * a.patch;
    p = p < 0 ? 0 : p > a.in_pixels - 1 ? a.in_pixels - 1 : p;   // (what such pixels hold is not used)
    g = g < M / 16 ? g : M / 16 - 1;
    block_request(a.x + ((int64_t)(p >> 5) * (M / 32) + (g >> 1)) * 1024 + (g & 1) * 512 + (p & 31) * 16, lds + L::patch + (uint32_t)k * 1024u);
  }

  // ---- the stream of filter fragments of this wavefront: 16 channels x 64 bytes of K each
  const int ca = M == 64 ? (wave & 3) : wave * CTA, pg = M == 64 ? wave >> 2 : 0;   // first channel tile (16) in A and C, group of pixels
  const int8_t* fa = a.wa + (ca >> 1) * TILE_A + (ca & 1) * 256;
  const int8_t* fb = a.wb + wave * UB * TILE_B;
  const int8_t* fc = a.wc + (ca >> 1) * TILE_C + (ca & 1) * 256;
  const int8_t* fs = KS ? a.ws + wave * UB * TILE_S : nullptr;
  const unsigned flane = (unsigned)((kg >> 1) * 1024 + (kg & 1) * 512 + col * 16);
  v4i ring[RING];
  auto fragment = [&](const int f) __attribute__((always_inline)) {
    if (f >= F) return;
    const int8_t* p;
    if (f < FA) p = fa + (f / CTA) * 2048 + (f % CTA) * 256;
    else if (f < FA + FS) p = fs + (f - FA) / (KS ? KS * 2 : 1) * TILE_S + (f - FA) / 2 % (KS ? KS : 1) * 2048 + ((f - FA) & 1) * 256;
    else if (f < FA + FS + FB) p = fb + (f - FA - FS) / (KA * 2) * TILE_B + (f - FA - FS) % KA * 2048 + ((f - FA - FS) / KA & 1) * 256;
    else p = fc + (f - FA - FS - FB) / (KC * CTA) * (M / 32) * TILE_C + (f - FA - FS - FB) / CTA % KC * 2048 + (f - FA - FS - FB) % CTA * 256;
    ring[f % RING] = *reinterpret_cast<const v4i*>(p + flane);
  };
#pragma unroll
  for (int f = 0; f < RING; ++f) fragment(f);

  // ---- the residual, or the pixels that its projection reads: behind the first fragments, which need not wait for them
  constexpr int RES = KS ? KS * NT / 8 : NT * M / 128;   // requests of every wavefront, at least
#pragma unroll
  for (int k = 0; k < (KS ? (KS * NT + 7) / 8 : RES); ++k) {
    const int part = (k * 8 + wave) * 4 + kg, g = part / NT;
    int p = p0 + (part - g * NT) * 16 + col;
    p = p > a.P - 1 ? a.P - 1 : p;
    if (KS) {
      int r, c, n;
      corner(p, r, c, n);
      p = (n * a.H + r + 1) * a.W + c + 1;
    }
    if (!KS || k * 8 + wave < KS * NT)
      block_request(a.res + ((int64_t)(p >> 5) * (KS ? KS * 2 : M / 8) + (g >> 1)) * 1024 + (g & 1) * 512 + (p & 31) * 16,
                    lds + (KS ? L::cut : L::wide) + (uint32_t)(k * 8 + wave) * 1024u);
  }
  if (tid < 4) *reinterpret_cast<v4i*>(block_lds + L::zero + tid * 16) = v4i{0, 0, 0, 0};

  // ---- windows of this lane's pixels: the byte of the first tap, and which of three rows and columns are inside
  int base[NTA], inside[NTA];
#pragma unroll
  for (int j = 0; j < NTA; ++j) {
    int p = p0 + (pg * NTA + j) * 16 + col, r, c, n;
    p = p > a.P - 1 ? a.P - 1 : p;
    corner(p, r, c, n);
    base[j] = L::patch + ((n * a.H + r) * a.W + c - first + kg * a.patch) * 16;
    inside[j] = 0;
#pragma unroll
    for (int t = 0; t < 9; ++t)
      inside[j] |= ((unsigned)(r + t / 3) < (unsigned)a.H && (unsigned)(c + t % 3) < (unsigned)a.W ? 1 : 0) << t;
  }
  block_landed<(RING < F ? RING : F) + RES>();   // biases and run
  block_barrier();

  // ---- A
  {
    v4i acc[CTA * NTA], b[2][NTA];
    auto operand = [&](const int step) __attribute__((always_inline)) {
      const int t = step / KA, k = step % KA, shift = ((t / 3) * a.W + t % 3 + k * 4 * a.patch) * 16;
#pragma unroll
      for (int j = 0; j < NTA; ++j) b[step & 1][j] = *reinterpret_cast<const v4i*>(block_lds + (inside[j] >> t & 1 ? base[j] + shift : L::zero));
    };
    operand(0);
#pragma unroll
    for (int i = 0; i < CTA; ++i)
#pragma unroll
      for (int j = 0; j < NTA; ++j) acc[i * NTA + j] = *reinterpret_cast<const v4i*>(block_lds + L::bias + ((ca + i) * 16 + kg * 4) * 4);
#pragma unroll
    for (int step = 0; step < 9 * KA; ++step) {
      if (step + 1 < 9 * KA) operand(step + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < CTA; ++i) {
#pragma unroll
        for (int j = 0; j < NTA; ++j)
          acc[i * NTA + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ring[(step * CTA + i) % RING], b[step & 1][j], acc[i * NTA + j], 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < CTA; ++i) fragment(step * CTA + i + RING);
      __builtin_amdgcn_sched_barrier(0);
    }
    block_settle(acc);
#pragma unroll
    for (int i = 0; i < CTA; ++i)
#pragma unroll
      for (int j = 0; j < NTA; ++j) {
        int v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = clamp_uniform(acc[i * NTA + j][e], a.qa.lo, a.qa.hi);
        *reinterpret_cast<uint32_t*>(block_lds + L::mid + (ca + i) * L::GROUP + ((pg * NTA + j) * 16 + col) * 16 + kg * 4) = shift_to_bytes(v[0], v[1], v[2], v[3], a.qa.shift);
      }
  }
  block_landed<(FA < F - RING ? FA : F > RING ? F - RING : 0)>();   // the residual: all but the fragments requested since
  block_barrier();

  // ---- the projection: to where the residual would have been fetched, every wavefront the channels that it adds
  if constexpr (KS > 0) {
#pragma unroll
    for (int u = 0; u < UB; ++u) {
      v4i acc[2 * NT];
      const int ct = (wave * UB + u) * 2;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i * NT + j] = *reinterpret_cast<const v4i*>(block_lds + L::bias + ((5 + UC) * M + (ct + i) * 16 + kg * 4) * 4);
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        v4i b[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) b[j] = *reinterpret_cast<const v4i*>(block_lds + L::cut + (k * 4 + kg) * L::GROUP + (j * 16 + col) * 16);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int f = FA + (u * KS + k) * 2 + i;
#pragma unroll
          for (int j = 0; j < NT; ++j) acc[i * NT + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ring[f % RING], b[j], acc[i * NT + j], 0, 0, 0);
          fragment(f + RING);
        }
      }
      block_settle(acc);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          int v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = clamp_uniform(acc[i * NT + j][e], a.qs.lo, a.qs.hi);
          *reinterpret_cast<uint32_t*>(block_lds + L::wide + (ct + i) * L::GROUP + (j * 16 + col) * 16 + kg * 4) = shift_to_bytes(v[0], v[1], v[2], v[3], a.qs.shift);
        }
    }
  }

  // ---- B: 16 channels after the other, all pixels; the result takes the residual's place.  The products of the next 16 run beside the requantisation.
  {
    v4i b[KA][NT], acc[2][NT];
#pragma unroll
    for (int k = 0; k < KA; ++k)
#pragma unroll
      for (int j = 0; j < NT; ++j) b[k][j] = *reinterpret_cast<const v4i*>(block_lds + L::mid + (k * 4 + kg) * L::GROUP + (j * 16 + col) * 16);
    int8_t* wide = block_lds + L::wide + wave * UB * 2 * L::GROUP + col * 16 + kg * 4;
    auto products = [&](const int u) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[u & 1][j] = *reinterpret_cast<const v4i*>(block_lds + L::bias + (M + (wave * UB * 2 + u) * 16 + kg * 4) * 4);
#pragma unroll
      for (int k = 0; k < KA; ++k) {
        const int f = FA + FS + u * KA + k;
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[u & 1][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ring[f % RING], b[k][j], acc[u & 1][j], 0, 0, 0);
        fragment(f + RING);
      }
    };
    products(0);
#pragma unroll
    for (int u = 0; u < 2 * UB; ++u) {
      uint32_t res[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j) res[j] = *reinterpret_cast<const uint32_t*>(wide + u * L::GROUP + j * 256);
      if (u + 1 < 2 * UB) products(u + 1);
      block_settle(acc[u & 1]);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        int v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = clamp_uniform(acc[u & 1][j][e], a.qb.lo, a.qb.hi) >> a.qb.shift;
          v[e] = clamp_uniform(wadd(v[e], (int32_t)(int8_t)(res[j] >> (8 * e))), a.qr.lo, a.qr.hi);
        }
        *reinterpret_cast<uint32_t*>(wide + u * L::GROUP + j * 256) = shift_to_bytes(v[0], v[1], v[2], v[3], a.qr.shift);
      }
    }
  }
  block_barrier();

  // ---- C
#pragma unroll
  for (int u = 0; u < UC; ++u) {
    v4i acc[CTA * NTA], b[2][NTA];
    const int ct = ca + u * (M / 16);
    const int8_t* at = block_lds + L::wide + kg * L::GROUP + (pg * NTA * 16 + col) * 16;
#pragma unroll
    for (int j = 0; j < NTA; ++j) b[0][j] = *reinterpret_cast<const v4i*>(at + j * 256);
#pragma unroll
    for (int i = 0; i < CTA; ++i)
#pragma unroll
      for (int j = 0; j < NTA; ++j) acc[i * NTA + j] = *reinterpret_cast<const v4i*>(block_lds + L::bias + (5 * M + (ct + i) * 16 + kg * 4) * 4);
#pragma unroll
    for (int k = 0; k < KC; ++k) {
#pragma unroll
      for (int j = 0; j < NTA; ++j)
        if (k + 1 < KC) b[(k + 1) & 1][j] = *reinterpret_cast<const v4i*>(at + (k + 1) * 4 * L::GROUP + j * 256);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < CTA; ++i) {
        const int f = FA + FS + FB + (u * KC + k) * CTA + i;
#pragma unroll
        for (int j = 0; j < NTA; ++j) acc[i * NTA + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ring[f % RING], b[k & 1][j], acc[i * NTA + j], 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < CTA; ++i) fragment(FA + FS + FB + (u * KC + k) * CTA + i + RING);
      __builtin_amdgcn_sched_barrier(0);
    }
    block_settle(acc);
#pragma unroll
    for (int i = 0; i < CTA; ++i)
#pragma unroll
      for (int j = 0; j < NTA; ++j) {
        int v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = clamp_uniform(acc[i * NTA + j][e], a.qc.lo, a.qc.hi);
        const uint32_t d = shift_to_bytes(v[0], v[1], v[2], v[3], a.qc.shift);
        const int p = p0 + (pg * NTA + j) * 16 + col, c = (ct + i) * 16;
        if (p < a.P)
          *reinterpret_cast<uint32_t*>(a.next + ((int64_t)(p >> 5) * (UC * M / 32) + (c >> 5)) * 1024 + ((c >> 4) & 1) * 512 + (p & 31) * 16 + kg * 4) = d;
      }
  }

  // ---- B's result to memory, 16 bytes of 16 neighbouring pixels a quarter of a wavefront
#pragma unroll
  for (int k = 0; k < NT * M / 128; ++k) {
    const int part = (k * 8 + wave) * 4 + kg, g = part / NT, p = p0 + (part - g * NT) * 16 + col;
    const v4i v = *reinterpret_cast<const v4i*>(block_lds + L::wide + (k * 8 + wave) * 1024 + lane * 16);
    if (p < a.P) *reinterpret_cast<v4i*>(a.out + ((int64_t)(p >> 5) * (M / 8) + (g >> 1)) * 1024 + (g & 1) * 512 + (p & 31) * 16) = v;
  }
}

static bool block_requant(const DevChain& c, bool bytes, BlockRequant* q) {
  return clamp_shift_of(c, &q->lo, &q->hi, &q->shift) && (!bytes || clamp_shift_narrow(q->lo, q->hi, q->shift));
}

// Pixels of the longest run of the input under `pixels` consecutive output pixels (the last tile's ends with the last pixel).
// How long a run is depends on where in its image the tile begins, and that comes again after OHW / gcd(OHW, pixels) tiles: 49 of 2 450 for
// 50 images of 56 x 56 and stride 2 in tiles of 16 (cvmhip_bottleneck_eligible with 128 channels 60 us of the host's time -> 4, 16 images 15 -> 3).
static int64_t block_run(int n, int h, int w, int oh, int ow, int stride, int pixels) {
  if (stride == 1) return pixels + 2 * (int64_t)w + 2;
  const int image = oh * ow, all = n * image, different = image / std::gcd(image, pixels);   // (32 bits: cvmhip_bottleneck_eligible)
  auto corner = [&](int p) {
    const int im = p / image, rem = p - im * image, r = rem / ow;
    return (int64_t)(im * h + r * stride - 1) * w + (rem - r * ow) * stride - 1;
  };
  int64_t most = 0;
  for (int k = 0, p = 0; k < different && p < all; ++k, p += pixels) {
    const int last = std::min(p + pixels, all) - 1;
    most = std::max(most, corner(last) + 2 * w + 2 - corner(p) + 1);
  }
  return most;
}

}  // namespace cvmhip

using namespace cvmhip;

namespace {

constexpr int64_t BLOCK_LDS_MOST = 160 * 1024;
constexpr int BLOCK_UNITS = 256;   // compute units

struct BlockForm { int nt; void (*kernel)(const BlockArgs); int64_t (*lds)(int64_t); void (*with_helpers)(const BlockArgs); };   // (lds: by the pixels of a run)
template <int M, int NT, int UC, int KS, int RING, int OCC>
BlockForm block_form() {
  BlockForm f = {NT, k_conv_block<M, NT, UC, KS, RING, OCC, false>, [](int64_t p) { return BlockLds<M, NT, UC, KS>::bytes(p); }, nullptr};
  if constexpr (M > 64 && NT == 1) f.with_helpers = k_conv_block<M, NT, UC, KS, RING, OCC, true>;
  return f;
}

// The smallest tile of which the chip holds all at once with one to a compute unit; where there are more, the last.  Microseconds a launch, filters of twelve
// layers in turn (tiles of 16, 32, 48 ... pixels):
//   M =  64, 56 x 56:  1 image 4.3 5.1 6.3 7.3 (32, 64, 96, 128), 4 images 6.7 5.9 7.0 8.0, 7 images 9.4 8.6 7.6 8.3, 16 images 21.2 15.9 16.5 15.4,
//                      50 images 54 37 33 31
//   M = 128, 28 x 28:  1 image 5.6 6.3 7.7 8.7 (16, 32, 48, 64), 7 images 8.7 6.8 8.1 9.3, 12 images 11.7 10.5 8.6 9.7, 16 images 14.6 11.0 12.7 10.3,
//                      24 images 20.6 16.3 15.7 17.4 and with 80 pixels 14.7, 50 images 40 27 27 26
//   M = 256, 14 x 14:  1 image 12.9 14.1 15.5 17.3 (16, 32, 48, 64), 16 images 12.9 13.7 15.6 17.5, 24 images 21 14.0 15.7 17.6, 50 images 35 28 20 22
// A number of fragments requested ahead between 9 and 40 makes no difference of more than 0.5.
constexpr int BLOCK_SIZES = 7;
#define BLOCK_SIZES_OF(UC, CUT)                                                                                                                   \
  {block_form<64, 2, UC, CUT, 15, 2>(), block_form<64, 4, UC, CUT, 12, 2>(), block_form<64, 6, UC, CUT, 6, 2>(),                                  \
   block_form<64, 8, UC, CUT, 6, 2>()},                                                                                                           \
  {block_form<128, 1, UC, 4 * CUT, 18, 2>(), block_form<128, 2, UC, 4 * CUT, 9, 2>(), block_form<128, 3, UC, 4 * CUT, 8, 2>(),                    \
   block_form<128, 4, UC, 4 * CUT, 8, 2>(), block_form<128, 5, UC, 4 * CUT, 12, 1>(), block_form<128, 6, UC, 4 * CUT, 12, 1>(),                   \
   block_form<128, 4, UC, 4 * CUT, 8, 2>()},                                                                                                      \
  {block_form<256, 1, UC, 8 * CUT, 14, 2>(), block_form<256, 2, UC, 8 * CUT, 18, 1>(), block_form<256, 3, UC, 8 * CUT, 12, 1>(),                  \
   block_form<256, 4, UC, 8 * CUT, 12, 1>()}
const BlockForm BLOCK_FORMS[3][3][BLOCK_SIZES] = {{BLOCK_SIZES_OF(1, 0)}, {BLOCK_SIZES_OF(2, 0)}, {BLOCK_SIZES_OF(1, 1)}};   // the last: with a projection
#undef BLOCK_SIZES_OF

const BlockForm* block_choose(int n, int m, int h, int w, int oc, int stride, bool projects, int* run) {
  const int oh = (h - 1) / stride + 1, ow = (w - 1) / stride + 1;
  const int64_t p = (int64_t)n * oh * ow;
  const BlockForm* best = nullptr;
  for (const BlockForm& f : BLOCK_FORMS[projects ? 2 : oc / m - 1][m == 64 ? 0 : m == 128 ? 1 : 2]) {
    if (f.nt == 0 || (best && p <= (int64_t)BLOCK_UNITS * 16 * best->nt)) break;
    const int64_t r = block_run(n, h, w, oh, ow, stride, 16 * f.nt);
    if (f.lds(r) > BLOCK_LDS_MOST) continue;   // (a stride of 2 has long runs)
    best = &f;
    *run = (int)r;
  }
  return best;
}

}  // namespace

extern "C" {

int cvmhip_bottleneck_eligible(int n, int m, int h, int w, int oc, int stride, const cvmhip_chain* chain_a, const cvmhip_chain* chain_b,
                               const cvmhip_chain* chain_r, const cvmhip_chain* chain_c, const cvmhip_bottleneck_projection* projection) {
  if (projection && (oc != m || projection->c != (m == 64 ? 64 : 2 * m))) return 0;
  if (n < 1 || (m != 64 && m != 128 && m != 256) || (oc != m && oc != 2 * m) || h < 1 || w < 1 || (stride != 1 && stride != 2)) return 0;
  if ((int64_t)n * h > INT32_MAX / 4 || (int64_t)n * h * w > INT32_MAX / 4 - 4096 || (int64_t)n * h * w * 4 * m > (int64_t)1 << 40) return 0;
  const cvmhip_chain* in[5] = {chain_a, chain_b, chain_r, chain_c, projection ? projection->chain : nullptr};
  for (int k = 0; k < (projection ? 5 : 4); ++k) {
    DevChain c;
    BlockRequant q;
    if (!make_chain(in[k], &c) || !block_requant(c, k != 1, &q)) return 0;
  }
  // The pixels that a projection reads take LDS beside the run of the input: where that leaves a smaller tile only, the projection is better a launch of its own
  // (50 images, M = 256 at 28 x 28 with stride 2: 42.7 us with tiles of 32 pixels, 24.0 with 48 and 17.6 for the projection).  Elsewhere: 16 images M = 64 15.2 us
  // against 15.5 + 7.2, M = 128 12.5 against 13.3 + 7.3, M = 256 18.0 against 13.9 + 7.5; 1 image 4.9 / 5.0 + 1, 6.4 / 6.2 + 4.0, 16.4 / 11.3 + 4.8.
  int run;
  const BlockForm* f = block_choose(n, m, h, w, oc, stride, projection != nullptr, &run);
  return f && (!projection || f->nt == block_choose(n, m, h, w, oc, stride, false, &run)->nt);
}

// us here / the layers in launches of their own, alone in a replayed graph with four sets of tensors in turn:
//   M = 256 of few pixels, where k_conv_run has the 3x3 layer and this launch 13 to 28 workgroups, each with all filters through its L1: 256 -> 256 at 8 x 8 13.6 / 11.1, 14 x 14 13.6 / 11.0, with the
//   projection 18.9 / 15.1, 512 out at 20 x 20 (400 pixels) 16.1 / 12.6; in a run of ResNet-50 (us with these blocks here / apart) 1 image 175.6 / 170.0, 2 (392 pixels) 178.3 / 174.2, 3 of
//   195 x 195 (507) 185.6 / 188.9, 4 (784) 196.0 / 199.4
//   Rows so long that LDS holds the run under a small tile only: M = 256, one 16-pixel tile where there would be two, 224 x 224 to 512 stride 2 58 / 44, 235 x 235 184 / 104, at best
//   138 x 138 stride 2 26 / 27; otherwise several rounds of tiles whose runs are many times as long: M = 64 at 702 x 702 stride 2 (68 pixels of a run to one of the tile) 69 / 42, 684 x 684 (34)
//   42.9 / 42.1, 654 x 654 with the projection (32.7) 40.6 / 52.6; M = 128 at 340 x 340 stride 2 (66) 50 / 36, 386 x 308 with the projection (31) 32 / 44, 328 x 516 stride 1 (33) 154 / 107, 326 x 454 (20) 116 / 101, 331 x 331 (11.4) 72.7 / 71.7,
//   319 x 319 (11.0) 63 / 69; M = 256 at 160 x 160 to 512 (11.1) 72 / 66
// Of 1 200 blocks drawn this keeps 126 apart, 91 of which were slower here than before there was this launch; of the others 2 are (2 %).
int cvmhip_bottleneck_gains(int n, int m, int h, int w, int oc, int stride, const cvmhip_bottleneck_projection* projection) {
  int run;
  const BlockForm* f = block_choose(n, m, h, w, oc, stride, projection != nullptr, &run);
  if (!f) return 0;
  const int64_t p = (int64_t)n * ((h - 1) / stride + 1) * ((w - 1) / stride + 1), round = (int64_t)BLOCK_UNITS * 16 * f->nt;
  if (m == 256 && (p <= 448 || (f->nt == 1 && p > round))) return 0;
  return p <= 3 * round || run <= (stride == 1 ? 11 : 33) * 16 * f->nt;
}

int cvmhip_conv2d_bottleneck_i8(const void* xp, const void* wa, const int32_t* bias_a, const cvmhip_chain* chain_a, const void* wb,
                                const int32_t* bias_b, const cvmhip_chain* chain_b, const void* residual, const cvmhip_chain* chain_r, void* out,
                                const void* wc, const int32_t* bias_c, const cvmhip_chain* chain_c, void* next, int n, int m, int h, int w, int oc,
                                int stride, const cvmhip_bottleneck_projection* projection, const cvmhip_bottleneck_filters* ahead, void* stream) {
  if (projection && (residual || !projection->w || !projection->x || (((uintptr_t)projection->w | (uintptr_t)projection->x | (uintptr_t)projection->bias) & 15)))
    return arg_error("conv2d_bottleneck_i8 projection");
  if (projection) residual = projection->x;
  if (!xp || !wa || !wb || !wc || !residual || !out || !next ||
      (((uintptr_t)bias_a | (uintptr_t)bias_b | (uintptr_t)bias_c | (uintptr_t)xp | (uintptr_t)wa | (uintptr_t)wb | (uintptr_t)wc | (uintptr_t)residual | (uintptr_t)out | (uintptr_t)next) & 15) ||
      !cvmhip_bottleneck_eligible(n, m, h, w, oc, stride, chain_a, chain_b, chain_r, chain_c, projection))
    return arg_error("conv2d_bottleneck_i8");
  BlockArgs a = {};
  DevChain c;
  make_chain(chain_a, &c); block_requant(c, true, &a.qa);
  make_chain(chain_b, &c); block_requant(c, false, &a.qb);
  make_chain(chain_r, &c); block_requant(c, true, &a.qr);
  make_chain(chain_c, &c); block_requant(c, true, &a.qc);
  if (projection) {
    make_chain(projection->chain, &c); block_requant(c, true, &a.qs);
    a.ws = reinterpret_cast<const int8_t*>(projection->w);
    a.bs = projection->bias;
  }
  a.x = reinterpret_cast<const int8_t*>(xp);
  a.wa = reinterpret_cast<const int8_t*>(wa);
  a.wb = reinterpret_cast<const int8_t*>(wb);
  a.wc = reinterpret_cast<const int8_t*>(wc);
  a.res = reinterpret_cast<const int8_t*>(residual);
  a.out = reinterpret_cast<int8_t*>(out);
  a.next = reinterpret_cast<int8_t*>(next);
  a.ba = bias_a; a.bb = bias_b; a.bc = bias_c;
  a.H = h; a.W = w; a.S = stride;
  const int oh = (h - 1) / stride + 1, ow = (w - 1) / stride + 1;
  a.OHW = oh * ow;
  a.OW = ow;
  a.P = n * oh * ow;
  a.in_pixels = n * h * w;
  a.div_ohw = make_fastdiv((uint32_t)a.OHW);
  a.div_ow = make_fastdiv((uint32_t)ow);
  const BlockForm* f = block_choose(n, m, h, w, oc, stride, projection != nullptr, &a.patch);
  a.div_patch = make_fastdiv((uint32_t)a.patch);
  a.tiles = (a.P + 16 * f->nt - 1) / (16 * f->nt);
  // The 1.1 MB of filters that a launch with M = 256 reads come from behind the L2 each time: all layers' are more than it holds.  Where most compute units
  // are idle some fetch the next launch's: ResNet-50, all blocks in one launch each, with 1 image 199.5 -> 193.3 us a run, 2 200.8 -> 196.1, 4 214.8 -> 211.9 (49 tiles); past that the
  // fetches are in the way (8 images 240.3 -> 241.2, 16 285 -> 288), and the question alone costs a launch 0.2 us, hence kernels of their own.
  if (ahead && ahead->m == 256 && f->with_helpers && a.tiles <= BLOCK_UNITS / 4) {
    a.helpers = 8;
    const int m2 = ahead->m;
    const void* filters[3] = {ahead->wa, ahead->wb, ahead->wc};
    const int kib[3] = {m2 / 32 * (9 * m2 / 32 + 1), m2 / 8 * (m2 / 32 + 1), ahead->oc / 32 * (m2 / 8 + 1)};
    for (int i = 0; i < 3; ++i) {
      a.ahead[i] = reinterpret_cast<const int8_t*>(filters[i]);
      a.ahead_kib[i] = filters[i] ? kib[i] : 0;
    }
  }
  char desc[128] = "";
  if (kernel_timing_enabled())
    snprintf(desc, sizeof(desc), "3x3/%d %d + 1x1 %d %s + 1x1 %d in %dx%dx%d out %dx%d tile %d grid %d + %d ahead", stride, m, 4 * m, projection ? "+ projection" : "+res", oc, n, h, w, oh, ow, 16 * f->nt, a.tiles, 8 * a.helpers);
  const double px = (double)a.P;
  const double cut = projection ? 4.0 * projection->c : 0.0;   // multiply-adds of the projection for a channel of m
  KernelTimer timer("k_conv_block", 2.0 * px * m * (9.0 * m + 4.0 * m + 4.0 * oc + cut), as_stream(stream),
                    (double)a.in_pixels * m + px * ((projection ? 4.0 * m + projection->c : 8.0 * m) + oc) + (double)m * (13.0 * m + 4.0 * oc + cut), desc);
  (a.helpers ? f->with_helpers : f->kernel)<<<(unsigned)(a.tiles + 8 * a.helpers), 512, (size_t)f->lds(a.patch), as_stream(stream)>>>(a);
  return check_launch("conv_block");
}

}  // extern "C"
