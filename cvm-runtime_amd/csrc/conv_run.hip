// 3 x 3 convolution, padding 1, stride 1 or 2, over a multiple of 128 channels of a pixel-blocked tensor with few pixels, int8 out, with or without the
// 2 x 2 max_pool2d behind it (the last stages of a ResNet and of a VGG, the extra layers of a detector).
//
// K is long and the pixels are few: k_conv_wave, which splits K over its wavefronts, sends each input byte through the L1 nine times, as much as or twice what
// the filter takes, in several trips to memory that nothing else covers.  Here a wavefront's share of K is 64 channels at a time: it fetches these of the run
// of input pixels under the workgroup's pixels into an LDS of its own, in the same trip the filter's fragments into registers, multiplies the taps from
// there, and no wavefront waits for another before the sums meet.  One trip to memory, the sums and the launch are what is left (512 -> 512 at 7 x 7:
// 7.2 -> 3.4 us); from some 100 output pixels on also the filter's way through the L1, 64 bytes a clock (16 images 8.9 -> 6.1).
//   workgroup: 16 * OT output channels x 16 * NT pixels; eight wavefronts with every eighth 64 channels each, or with every fourth or second and some of the
//   taps where there are fewer channels
// The pixels lie granule by granule in LDS, so that sixteen neighbours are one read of 256 bytes; a tap outside the image reads sixteen zeros.
// v_mfma_i32_16x16x64_i8 with the filter as first operand.
#include <algorithm>

#include "conv_mfma.h"
#include "requant.h"

namespace cvmhip {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int RUN_SLICE = 19 * 1024;                     // LDS of a wavefront's pixels
constexpr int RUN_PIXELS = RUN_SLICE / 64;
constexpr int RUN_BIAS = 64, RUN_DATA = 64 + 256;        // 64 zeros, the bias of up to 64 channels, then slices or sums
constexpr int RUN_LDS = RUN_DATA + 8 * RUN_SLICE;

struct RunArgs {
  const int8_t* x;
  const int8_t* wf;
  int8_t* out;
  const int32_t* bias;
  int H, W, S, C, units, in_pixels, OHW, OW;   // units: output pixels of all images; OHW, OW of one
  int run, oblocks;                            // pixels of the longest run under a tile; output channels in tiles of 32
  int lo, hi, shift, tile_bytes, octiles;      // tile_bytes: from 32 filter rows to the next
  FastDiv div_oc, div_ohw, div_ow, div_run;
};

__device__ __forceinline__ int run_min(int a, int b) { return a < b ? a : b; }

// One request of 64 x 16 bytes.  The LDS it writes has been read: the reads before it have returned.
__device__ __forceinline__ void run_request(const void* from, uint32_t lds_at) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(from), "s"(lds_at) : "memory");
}

// TG: wavefronts that share 64 channels, by taps (1: nine taps each, 2: five or four, 4: three or two); AHEAD: taps whose fragments are in registers
template <int OT, int NT, bool POOL, int TG, int AHEAD>
__global__ void __launch_bounds__(512, 2) k_conv_run(const RunArgs a) {
  constexpr int WAYS = 8 / TG, TAPS = (9 + TG - 1) / TG;
  static_assert(AHEAD <= TAPS, "");
  constexpr int UNITS = POOL ? 4 * NT : 16 * NT;   // pixels of the output; with the pool tile j is corner j % 4 of sixteen windows
  static_assert(!POOL || NT % 4 == 0, "four corners of sixteen windows");
  __shared__ __attribute__((aligned(16))) int8_t run_lds[RUN_LDS];
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, kg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) int8_t*)run_lds;
  const int group = (int)fastdiv(blockIdx.x, a.div_oc), oc0 = ((int)blockIdx.x - group * a.octiles) * (16 * OT);
  const int u0 = group * UNITS;
  const int bias = a.bias && tid < 16 * OT ? a.bias[oc0 + tid] : 0;
  auto corner = [&](int u, int& n, int& row, int& column) __attribute__((always_inline)) {   // of the 3 x 3 window in the input
    n = (int)fastdiv((unsigned)u, a.div_ohw);
    const int rem = u - n * a.OHW, y = (int)fastdiv((unsigned)rem, a.div_ow);
    row = y * a.S - 1;
    column = (rem - y * a.OW) * a.S - 1;
  };
  int first;
  {
    int n, r, c;
    corner(u0, n, r, c);
    first = (n * a.H + r) * a.W + c;
  }
  int window[NT];   // LDS address of a pixel's window (a multiple of 16) << 5, and which of its taps lie in the image
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    int u = u0 + (POOL ? j >> 2 : j) * 16 + col, n, r, c;
    u = u < a.units ? u : a.units - 1;
    corner(u, n, r, c);
    if (POOL) {
      r += j >> 1 & 1;
      c += j & 1;
    }
    window[j] = (RUN_DATA + wave * RUN_SLICE + ((n * a.H + r) * a.W + c - first + kg * a.run) * 16) << 5;
#pragma unroll
    for (int t = 0; t < 9; ++t) window[j] |= ((unsigned)(r + t / 3) < (unsigned)a.H && (unsigned)(c + t % 3) < (unsigned)a.W ? 1 : 0) << t;
  }
  if (tid < 4) *reinterpret_cast<v4i*>(run_lds + tid * 16) = v4i{0, 0, 0, 0};
  const unsigned granule = (unsigned)((kg >> 1) * 1024 + (kg & 1) * 512 + col * 16);
  auto fragment = [&](int i, int chunk) __attribute__((always_inline)) {   // 16 output channels, KiB of the filter before it
    const int ot = (oc0 >> 4) + i;
    const int8_t* at = a.wf + ((int64_t)(ot >> 1) * a.tile_bytes + (ot & 1) * 256 + (int64_t)chunk * 1024);
    return *reinterpret_cast<const v4i*>(at + granule);
  };
  v4i acc[OT][NT];
#pragma unroll
  for (int i = 0; i < OT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = v4i{0, 0, 0, 0};
  const int requests = (4 * a.run + 63) >> 6, tap_chunks = a.C / 32;
  __syncthreads();   // the zeros
  const int share = wave % WAYS, tap0 = wave / WAYS * 9 / TG, taps = (wave / WAYS + 1) * 9 / TG - tap0;
  for (int c64 = share; c64 < a.C / 64; c64 += WAYS) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    for (int k = 0; k < requests; ++k) {
      const int t = k * 64 + lane;
      int g = (int)fastdiv((unsigned)t, a.div_run), p = first + t - g * a.run;
      p = p < 0 ? 0 : p > a.in_pixels - 1 ? a.in_pixels - 1 : p;   // (outside the tensor, or behind the run: not used)
      g = g < 4 ? g : 3;
      run_request(a.x + ((int64_t)(p >> 5) * (a.C / 32) + c64 * 2 + (g >> 1)) * 1024 + (g & 1) * 512 + (p & 31) * 16,
                  lds + (uint32_t)(RUN_DATA + wave * RUN_SLICE + k * 1024));
    }
    v4i f[AHEAD][OT];
#pragma unroll
    for (int t = 0; t < AHEAD; ++t)
#pragma unroll
      for (int i = 0; i < OT; ++i) f[t][i] = fragment(i, (tap0 + run_min(t, taps - 1)) * tap_chunks + c64 * 2);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AHEAD * OT) : "memory");   // the pixels, which this wavefront alone reads
#pragma unroll
    for (int t = 0; t < TAPS; ++t) {
      const int tap = TG == 1 ? t : tap0 + t, at = ((tap / 3) * a.W + tap % 3) * 16;
#pragma unroll
      for (int j = 0; j < NT; ++j) asm volatile("" : "+v"(window[j]));   // (or the addresses of all taps are worked out in front of the loop)
      v4i b[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j) b[j] = *reinterpret_cast<const v4i*>(run_lds + ((TG == 1 || t < taps) && (window[j] >> tap & 1) ? (window[j] >> 5 & ~15) + at : 0));
#pragma unroll
      for (int i = 0; i < OT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f[t % AHEAD][i], b[j], acc[i][j], 0, 0, 0);
      if (t + AHEAD < TAPS)
#pragma unroll
        for (int i = 0; i < OT; ++i) f[t % AHEAD][i] = fragment(i, (tap0 + run_min(t + AHEAD, taps - 1)) * tap_chunks + c64 * 2);
      if (OT * NT == 32) __builtin_amdgcn_sched_barrier(0);   // (reads of a tap ahead would spill)
    }
  }
  // the wavefronts' sums meet, at most 128 KB at a time
  constexpr int ROWS = OT * NT <= 16 ? OT : 16 / NT;
#pragma unroll
  for (int i0 = 0; i0 < OT; i0 += ROWS) {
    __syncthreads();   // slices or sums have been read
    if (i0 == 0 && tid < 16 * OT) reinterpret_cast<int*>(run_lds + RUN_BIAS)[tid] = bias;
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) *reinterpret_cast<v4i*>(run_lds + RUN_DATA + ((wave * ROWS + i) * NT + j) * 1024 + lane * 16) = acc[i0 + i][j];
    __syncthreads();
    constexpr int TILES = POOL ? ROWS * NT / 4 : ROWS * NT;   // of sixteen channels x sixteen stored pixels
#pragma unroll
    for (int k = 0; k < (TILES + 7) / 8; ++k) {
      const int tile = k * 8 + wave;
      if (TILES % 8 && tile >= TILES) break;
      const int i = POOL ? tile / (NT / 4 ? NT / 4 : 1) : tile / NT, j = POOL ? tile % (NT / 4 ? NT / 4 : 1) : tile % NT;
      const int8_t* at = run_lds + RUN_DATA + (i * NT + (POOL ? 4 * j : j)) * 1024 + lane * 16;
      const v4i bv = *reinterpret_cast<const v4i*>(run_lds + RUN_BIAS + ((i0 + i) * 16 + kg * 4) * 4);
      v4i most;
#pragma unroll
      for (int q = 0; q < (POOL ? 4 : 1); ++q) {
        v4i sum = bv;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
          const v4i v = *reinterpret_cast<const v4i*>(at + (s * ROWS * NT + q) * 1024);
#pragma unroll
          for (int e = 0; e < 4; ++e) sum[e] = wadd(sum[e], v[e]);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) most[e] = q == 0 ? sum[e] : max(most[e], sum[e]);   // (clamp and shift never fall as their input grows)
      }
      const uint32_t d = shift_to_bytes(clamp_uniform(most[0], a.lo, a.hi), clamp_uniform(most[1], a.lo, a.hi), clamp_uniform(most[2], a.lo, a.hi),
                                        clamp_uniform(most[3], a.lo, a.hi), a.shift);
      const int p = u0 + j * 16 + col, oc = oc0 + (i0 + i) * 16;
      if (p < a.units) *reinterpret_cast<uint32_t*>(a.out + ((int64_t)(p >> 5) * a.oblocks + (oc >> 5)) * 1024 + ((oc >> 4) & 1) * 512 + (p & 31) * 16 + kg * 4) = d;
    }
  }
}

struct RunForm { int ot, nt; };
static const RunForm RUN_FORMS[] = {{1, 1}, {1, 2}, {2, 2}, {2, 4}, {4, 4}}, RUN_POOL_FORMS[] = {{1, 4}, {2, 4}, {4, 4}, {4, 8}};

// pixels of the longest run of input under a tile of `units` output pixels
static int run_length(const RunArgs& a, bool pool, int units) {   // (32 bits: the tensor has fewer bytes than that; at most 256 tiles)
  auto corner = [&](int u) {
    const int n = u / a.OHW, rem = u % a.OHW;
    return (n * a.H + rem / a.OW * a.S - 1) * a.W + rem % a.OW * a.S - 1;
  };
  int most = 0;
  for (int u = 0; u < a.units; u += units) most = std::max(most, corner(std::min(u + units, a.units) - 1) - corner(u));
  return most + (pool ? 3 : 2) * (a.W + 1) + 1;
}

// Layers for which k_conv_wave, whose workgroups are larger, is ahead.  What a workgroup here fetches of each input channel, the run once for every wavefront
// that shares the channel and the filter, goes through its L1; us with k_conv_wave / here, output pixels and these bytes (2 200 layers drawn: 183 were slower here; of 1 500 others that it still takes 31 are, 12 by more than 5 %):
//   384, 640, 896 channels (several shares in turn, four wavefronts to each): 384 at 3 x 41 x 41 to 128 stride 2 (1 323, 1 196) 7.0 / 9.4, 896 at 37 x 37 to 64 (1 369, 576) 9.4 / 11.1, at 2 x 26 x 38
//   to 64 stride 2 (494, 732) 9.7 / 11.9, at 2 x 40 x 40 to 192 stride 2 (800, 1 188) 14.5 / 17.0; below: 384 at 30 x 30 to 256 (900, 664) 7.4 / 6.5, at 12 x 15 x 15 to 256 stride 2 (768, 836) 9.2 / 7.8
//   256 and 768 (two): 256 at 16 x 25 x 25 to 128 stride 2 (2 704, 886) 6.3 / 8.1, 768 at 39 x 45 to 192 (1 755, 600) 10.7 / 11.7; below: 256 at 12 x 13 x 13 to 128 (2 028, 408) 6.0 / 4.6, at
//   45 x 45 to 128 in 32 x 32 tiles (2 025, 536) 6.0 / 5.2
//   512 and its multiples, tiles of 64 pixels: 512 to 128 at 6 144 pixels 9.0 / 10.1, to 256 at 3 600 9.7 / 10.5, 1024 to 128 at 6 720 15.2 / 16.2; below: 512 to 512 at 1 849 10.3 / 10.0; long runs under
//   16 x 32 tiles: 512 to 64 stride 2 at 1 352 (331) 7.5 / 8.3; with the pool in 32 x 64 tiles, 512 to 128 at 1 444 9.9 / 10.7, in 64 x 128 at 2 592 15.8 / 13.9
static bool run_falls_behind(int c, int oc, int form, int ot, bool pool, const RunArgs& a) {
  const int wavefronts = c % 512 == 0 ? 1 : c % 256 == 0 ? 2 : 4, bytes = wavefronts * a.run + 9 * 16 * ot;
  if (pool) return c == 512 && form == 2 && a.units > 1000;
  if (wavefronts == 1) return (form >= 3 && a.units > 4 * c) || (c == 512 && form == 1 && a.units > 1000 && bytes > 300);
  if (wavefronts == 2) return a.units > 950 && bytes > (form == 2 && c == 256 ? 620 : 484);
  return wavefronts == 4 && c > 128 && (a.units > 1200 || bytes > (oc <= 192 ? 600 : 950));
}

// Which form takes the layer, -1: none.  (g and ep as conv_prepare leaves them; fills `a`)
// The smallest tile that makes one round of workgroups, one to a compute unit; us with k_conv_wave / here, one layer again and again in a replayed graph
// with four sets of operands in turn (in a run of a model, by its events: 16 images at 7 x 7 8.1 / 6.8, at 14 x 14 with the pool 15.6 / 14.9):
//   512 -> 512 at 7 x 7: 1 image 7.2 / 3.4, 3 7.7 / 4.2, 8 8.7 / 4.9, 16 8.9 / 6.1, 24 9.9 / 8.1, 32 9.9 / 8.8; 50, which would be 64 x 128, 14.0 / 14.0
//   at 14 x 14: 1 8.4 / 4.4, 8 10.0 / 8.9, 16 (64 x 128) 14.5 / 14.6; with the pool 1 8.9 / 5.7, 8 10.3 / 8.9, 16 (64 x 128) 14.9 / 13.4; stride 2 1 7.4 / 3.7, 16 12.7 / 8.5
//   256 channels (taps dealt to two): 1 x 7 x 7 5.8 / 3.5, 4 x 14 x 14 6.0 / 4.6, 8 x 14 x 14 (32 x 64) 6.2 / 5.8, 768 at 4 x 14 x 14 10.6 / 7.2
//   128 (to four): 1 x 8 x 8 to 256 stride 2 5.1 / 3.4, 2 x 28 x 28 5.3 / 4.4; 32 x 64 would be 5.4 / 5.8 at 1 x 56 x 56, 5.6 / 5.6 at 8 x 28 x 28
// So 64 x 128 only with the pool, 64 x 64 only where a wavefront has all nine taps, 32 x 64 not where it has three.
static int run_choose(const ConvGeom& g, const Epilogue& ep, RunArgs* a) {
  if (g.dw || g.row_bytes || g.Cp % (ep.pool ? 512 : 128) != 0 || g.OC % 64 != 0 || g.KH != 3 || g.KW != 3 || g.SH != g.SW || g.SH < 1 || g.SH > 2 || g.PH != 1 || g.PW != 1 ||
      g.DH != 1 || g.DW != 1 || ep.out_mode != OUT_I8_ACT || ep.out_cp != g.OC || ep.residual || ep.split || (ep.pool && g.SH != 1))
    return -1;
  if ((int64_t)g.N * g.H * g.W * g.Cp > INT32_MAX || !clamp_shift_of(ep.chain, &a->lo, &a->hi, &a->shift) || !clamp_shift_narrow(a->lo, a->hi, a->shift)) return -1;
  const bool pool = ep.pool != 0;
  a->H = g.H; a->W = g.W; a->C = g.Cp;
  a->S = pool ? 2 : g.SH;
  a->OW = pool ? g.OW / 2 : g.OW;
  a->OHW = pool ? g.OH / 2 * a->OW : g.OH * g.OW;
  a->units = g.N * a->OHW;
  a->in_pixels = g.N * g.H * g.W;
  const RunForm* forms = pool ? RUN_POOL_FORMS : RUN_FORMS;
  for (int f = 0; f < (pool ? 4 : g.Cp % 512 == 0 ? 5 : g.Cp % 256 == 0 ? 4 : 3); ++f) {
    const int units = pool ? 4 * forms[f].nt : 16 * forms[f].nt;
    if ((int64_t)((a->units + units - 1) / units) * (g.OC / (16 * forms[f].ot)) > 256) continue;
    a->run = run_length(*a, pool, units);
    return a->run > RUN_PIXELS || run_falls_behind(g.Cp, g.OC, f, forms[f].ot, pool, *a) ? -1 : f;
  }
  return -1;
}

int64_t conv_run_blocks(const ConvGeom& g, const Epilogue& ep) {
  RunArgs a = {};
  const int f = run_choose(g, ep, &a);
  if (f < 0) return 0;
  const RunForm& form = (ep.pool ? RUN_POOL_FORMS : RUN_FORMS)[f];
  const int units = ep.pool ? 4 * form.nt : 16 * form.nt;
  return (int64_t)((a.units + units - 1) / units) * (g.OC / (16 * form.ot));
}

int conv_run(const int8_t* xp, const int8_t* wp, void* out, const ConvGeom& g, const Epilogue& ep, hipStream_t s) {
  RunArgs a = {};
  const int f = run_choose(g, ep, &a);
  if (f < 0) return arg_error("conv_run");
  const RunForm& form = (ep.pool ? RUN_POOL_FORMS : RUN_FORMS)[f];
  a.x = xp;
  a.wf = wp;
  a.out = reinterpret_cast<int8_t*>(out);
  a.bias = ep.bias;
  a.oblocks = g.OC / 32;
  a.tile_bytes = (g.Kp / 32 + 1) * 1024;
  a.octiles = g.OC / (16 * form.ot);
  a.div_oc = make_fastdiv((uint32_t)a.octiles);
  a.div_ohw = make_fastdiv((uint32_t)a.OHW);
  a.div_ow = make_fastdiv((uint32_t)a.OW);
  a.div_run = make_fastdiv((uint32_t)a.run);
  const bool pool = ep.pool != 0;
  const int units = (pool ? 4 : 16) * form.nt;
  const unsigned grid = (unsigned)((a.units + units - 1) / units * a.octiles);
#define RUN_CASE(OT, NT, POOL, TG, AHEAD) k_conv_run<OT, NT, POOL, TG, AHEAD><<<grid, 512, 0, s>>>(a)
  if (pool && f == 0) RUN_CASE(1, 4, true, 1, 9);
  else if (pool && f == 1) RUN_CASE(2, 4, true, 1, 9);
  else if (pool && f == 2) RUN_CASE(4, 4, true, 1, 9);
  else if (pool) RUN_CASE(4, 8, true, 1, 4);
  else if (g.Cp % 256 != 0) {
    if (f == 0) RUN_CASE(1, 1, false, 4, 3);
    else if (f == 1) RUN_CASE(1, 2, false, 4, 3);
    else RUN_CASE(2, 2, false, 4, 3);
  } else if (g.Cp % 512 != 0) {
    if (f == 0) RUN_CASE(1, 1, false, 2, 5);
    else if (f == 1) RUN_CASE(1, 2, false, 2, 5);
    else if (f == 2) RUN_CASE(2, 2, false, 2, 5);
    else RUN_CASE(2, 4, false, 2, 5);
  } else if (f == 0) RUN_CASE(1, 1, false, 1, 9);
  else if (f == 1) RUN_CASE(1, 2, false, 1, 9);
  else if (f == 2) RUN_CASE(2, 2, false, 1, 9);
  else if (f == 3) RUN_CASE(2, 4, false, 1, 9);
  else RUN_CASE(4, 4, false, 1, 9);
#undef RUN_CASE
  return check_launch("conv_run");
}

}  // namespace cvmhip

using namespace cvmhip;

extern "C" int cvmhip_conv2d_run_eligible(const cvmhip_chain* chain, int n, int ic, int h, int w, int oc, int kh, int kw, int stride_h, int stride_w,
                                          int pad_h, int pad_w, int dil_h, int dil_w) {
  if (n < 1 || ic < 1 || ic % 128 != 0 || oc < 1 || h < 1 || w < 1 || kh != 3 || kw != 3 || pad_h != 1 || pad_w != 1 || stride_h < 1 || stride_w < 1) return 0;
  if ((int64_t)n * h > INT32_MAX || (int64_t)n * h * w > INT32_MAX || (int64_t)n * h * w * ic > INT32_MAX) return 0;   // (as cvmhip_conv2d_i8 refuses them)
  ConvGeom g = {};
  Epilogue ep = {};
  if (!make_chain(chain, &ep.chain)) return 0;
  g.N = n; g.H = h; g.W = w; g.Cp = ic; g.OC = oc;
  g.OH = (h - 1) / stride_h + 1; g.OW = (w - 1) / stride_w + 1;
  g.KH = kh; g.KW = kw; g.SH = stride_h; g.SW = stride_w; g.PH = pad_h; g.PW = pad_w; g.DH = dil_h; g.DW = dil_w;
  ep.out_mode = OUT_I8_ACT;
  ep.out_cp = oc;
  RunArgs a = {};
  return conv_run_blocks(g, ep) <= 0 ? 0 : g.Cp % 512 == 0 && run_choose(g, ep, &a) == 0 ? 2 : 1;
}
