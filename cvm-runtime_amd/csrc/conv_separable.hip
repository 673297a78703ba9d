// Depthwise 3x3 convolution and the 1x1 convolution that reads it, one launch for both.
//
// At one image these layers of a MobileNet are bound by the launch: each is 4 to 5 us of which 1.3 are the launch itself and
// the rest a chain of addresses, first operands from behind a cold L2, a few products and a store, whose result the next
// launch fetches again.  Here a workgroup of eight wavefronts computes the depthwise result of a tile of pixels for ALL
// channels into LDS, in the fragment order of the second convolution's operand, and multiplies it from there.  The depthwise
// tensor never reaches memory.
//   tile: 32 * WP pixels x 32 * WO output channels, WO * WP = 8 wavefronts.  With more output channels than 256 several
//   workgroups compute the same depthwise tile, whose products are a few percent of the 1x1 part's.
// Depthwise part: v_mfma_i32_32x32x32_i8 with the diagonal matrix of a tap's 32 weights, which every lane makes from the
// twelve bytes of its channel (a filter packed as diagonals is nine times the bytes); padding taps read past the buffer
// (zero).  The first filter fragments of the 1x1 part are requested before it.
// Measured on SSD-512, two launches against one: 256 x 256 x 32 -> 64 12.6 and 8.0 us, 128 x 128 x 128 -> 128 11.1 and 5.5, 32 x 32
// x 512 -> 512 8.7 and 6.4.  What bounds it now: instructions and the latency of two dependent fetches (of 13 K clocks of a
// 512-channel tile 2 K are the places of the taps, 1.2 K the first operands' way, 2 K each of two depthwise units on two
// wavefronts to a SIMD, 1.7 K the products); three loads and shifts between lanes instead of nine loads, requesting the
// next unit's operands ahead, and half or a quarter of the output channels per workgroup with K cut in as many shares all took
// 0.3 to 1 us longer.
#include <string.h>

#include "conv_mfma.h"
#include "requant.h"

namespace cvmhip {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v3i __attribute__((ext_vector_type(3)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

// a chain, and its values if it is one clamp and shift
struct SepChain {
  DevChain chain;
  int plain, lo, hi, shift;
};
struct SepArgs {
  const int8_t* x;         // act tensor, C channels
  const uint32_t* wd;      // [channel][3 dwords]: the nine weights
  const int32_t* bd;
  const int8_t* wf;        // packed filter of the 1x1 convolution
  const int32_t* bp;
  int8_t* out;             // act tensor, OC channels
  int H, W, OH, OW, SH, SW, PH, PW;
  int P, ktiles, octiles, nch1, otgroups;
  unsigned x_bytes;
  FastDiv div_ohw, div_ow, div_groups;
  SepChain first, second;
};

constexpr int SEP_WAVES = 8;
constexpr int SEP_AHEAD = 8;         // filter fragments in flight
constexpr size_t SEP_LDS_MOST = 64 * 1024;   // of the depthwise tile

__device__ __forceinline__ void sep_chain(const SepChain& c, int32_t (&v)[16]) {
  if (c.plain) {
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = clamp_uniform(v[e], c.lo, c.hi) >> c.shift;
    return;
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    if (t >= c.chain.count) break;
    const DevStage s = c.chain.st[t];
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = apply_stage(s, v[e]);
  }
}
// the 16 values of a lane are channels 8q + 4 (lane >> 5) .. + 3, q = 0 .. 3
__device__ __forceinline__ void sep_bias(const int32_t* bias, int c0, int lgrp, v4i (&v)[4]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = bias ? *reinterpret_cast<const v4i*>(bias + c0 + q * 8 + lgrp * 4) : v4i{0, 0, 0, 0};
}

template <int WO>
__global__ void __launch_bounds__(512) k_conv_separable(const SepArgs a) {
  constexpr int WP = SEP_WAVES / WO;
  extern __shared__ __attribute__((aligned(16))) int8_t sep_lds[];   // [channel tile][pixel block][1 KiB fragment]
  const int tid = threadIdx.x, lane = tid & 63, lrow = lane & 31, lgrp = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ptile = (int)fastdiv(blockIdx.x, a.div_groups), group = (int)blockIdx.x - ptile * a.otgroups;
  const int px0 = ptile * (32 * WP);

  // ---- first fragments of the 1x1 filter
  const int ot = group * WO + wave % WO, wp = wave / WO;
  const bool active = ot < a.octiles && px0 + wp * 32 < a.P;
  const int8_t* wf = a.wf + ((int64_t)(ot < a.octiles ? ot : 0) * a.nch1) * 1024 + lane * 16;
  v4i fa[SEP_AHEAD];
#pragma unroll
  for (int k = 0; k < SEP_AHEAD; ++k) fa[k] = *reinterpret_cast<const v4i*>(wf + (k < a.ktiles ? k : 0) * 1024);
  v4i bias[4];
  sep_bias(a.bp, (ot < a.octiles ? ot : 0) * 32, lgrp, bias);

  // ---- depthwise: this wavefront's pixel block, every WO-th channel tile
  {
    const int pb = wave % WP, p = px0 + pb * 32 + lrow;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(a.x), 0, (int)a.x_bytes, 0x00020000);
    int off[9];
    {
      const unsigned pp = p < a.P ? (unsigned)p : 0u;
      const int n = (int)fastdiv(pp, a.div_ohw), rem = (int)pp - n * (a.OH * a.OW), oh = (int)fastdiv((unsigned)rem, a.div_ow), ow = rem - oh * a.OW;
      const int ih0 = oh * a.SH - a.PH, iw0 = ow * a.SW - a.PW;
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        const int ih = ih0 + t / 3, iw = iw0 + t % 3;
        const unsigned pin = (unsigned)((n * a.H + ih) * a.W + iw);
        const bool ok = (unsigned)ih < (unsigned)a.H && (unsigned)iw < (unsigned)a.W;
        off[t] = ok ? (int)((pin >> 5) * (unsigned)a.ktiles * 1024u + (pin & 31u) * 16u + (unsigned)lgrp * 512u) : 0x7f000000;
      }
    }
    // the byte of a fragment row that lies on the diagonal
    int mask[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) mask[d] = (lrow >> 4) == lgrp && ((lrow & 15) >> 2) == d ? 0xff << (8 * (lrow & 3)) : 0;
    for (int kt = wave / WP; kt < a.ktiles; kt += WO) {
      v4i x[9], bd[4];
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        const v4u v = __builtin_amdgcn_raw_buffer_load_b128(rs, off[t], kt * 1024, 0);
        x[t] = v4i{(int)v[0], (int)v[1], (int)v[2], (int)v[3]};
      }
      const v3i w = *reinterpret_cast<const v3i*>(a.wd + (unsigned)(kt * 32 + lrow) * 3u);
      sep_bias(a.bd, kt * 32, lgrp, bd);
      v16i acc;
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[e] = bd[e >> 2][e & 3];
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        const int all = (int)__builtin_amdgcn_perm(0u, (uint32_t)w[t / 4], 0x01010101u * (t & 3));
        const v4i diag = {all & mask[0], all & mask[1], all & mask[2], all & mask[3]};
        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(diag, x[t], acc, 0, 0, 0);
      }
      asm volatile(WAIT_16_PASSES : "+v"(acc));
      int32_t v[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) v[e] = acc[e];
      sep_chain(a.first, v);
      int8_t* f = sep_lds + (kt * WP + pb) * 1024 + lrow * 16 + lgrp * 4;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<uint32_t*>(f + (q >> 1) * 512 + (q & 1) * 8) = low_bytes(v[q * 4], v[q * 4 + 1], v[q * 4 + 2], v[q * 4 + 3]);
    }
  }
  __syncthreads();
  if (!active) return;

  // ---- 1x1: one tile of 32 channels x 32 pixels per wavefront
  v16i acc[2];
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    acc[0][e] = bias[e >> 2][e & 3];
    acc[1][e] = 0;
  }
  const int8_t* f = sep_lds + wp * 1024 + lane * 16;
  for (int k0 = 0; k0 < a.ktiles; k0 += SEP_AHEAD) {
    v4i b[SEP_AHEAD];
#pragma unroll
    for (int k = 0; k < SEP_AHEAD; ++k)
      if (k0 + k < a.ktiles) b[k] = *reinterpret_cast<const v4i*>(f + (k0 + k) * (WP * 1024));
#pragma unroll
    for (int k = 0; k < SEP_AHEAD; ++k) {
      if (k0 + k < a.ktiles) acc[k & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[k], b[k], acc[k & 1], 0, 0, 0);
      const int next = k0 + SEP_AHEAD + k;
      if (k0 + SEP_AHEAD < a.ktiles) fa[k] = *reinterpret_cast<const v4i*>(wf + (next < a.ktiles ? next : 0) * 1024);
    }
  }
  int32_t v[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) v[e] = wadd(acc[0][e], acc[1][e]);
  sep_chain(a.second, v);
  uint32_t d[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) d[q] = low_bytes(v[q * 4], v[q * 4 + 1], v[q * 4 + 2], v[q * 4 + 3]);
  const v4i w = sixteen_channels(d);
  const int p = px0 + wp * 32 + lrow;
  if (p < a.P) *reinterpret_cast<v4i*>(a.out + ((int64_t)(p >> 5) * a.octiles + ot) * 1024 + lane * 16) = w;
}

__global__ void __launch_bounds__(256) k_pack_separable(const int32_t* __restrict__ w, uint32_t* __restrict__ wd, int channels) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= channels) return;
  uint32_t d[3] = {0, 0, 0};
  for (int t = 0; t < 9; ++t) d[t >> 2] |= (uint32_t)(uint8_t)(int8_t)w[c * 9 + t] << (8 * (t & 3));
  for (int k = 0; k < 3; ++k) wd[c * 3 + k] = d[k];
}

static SepChain sep_chain_of(const DevChain& c) {
  SepChain s = {c, 0, 0, 0, 0};
  s.plain = clamp_shift_of(c, &s.lo, &s.hi, &s.shift);
  return s;
}

}  // namespace cvmhip

using namespace cvmhip;

extern "C" {

size_t cvmhip_separable_filter_bytes(int c) { return (size_t)c * 12; }

int cvmhip_pack_separable_filter(const int32_t* w, void* wd, int c, void* stream) {
  if (!w || !wd || ((uintptr_t)wd & 15) || c < 1) return arg_error("pack_separable_filter");
  k_pack_separable<<<(unsigned)((c + 255) / 256), 256, 0, as_stream(stream)>>>(w, reinterpret_cast<uint32_t*>(wd), c);
  return check_launch("pack_separable_filter");
}

// output channel tiles per workgroup: as many as the layer has, up to all eight wavefronts
static int sep_wo(int octiles) { return octiles >= 8 ? 8 : octiles >= 4 ? 4 : octiles >= 2 ? 2 : 1; }

int cvmhip_separable_eligible(int n, int c, int h, int w, int oc, int stride_h, int stride_w, int pad_h, int pad_w) {
  if (n < 1 || c < 32 || (c % 32) != 0 || oc < 32 || (oc % 32) != 0 || h < 1 || w < 1 || stride_h < 1 || stride_w < 1 || pad_h < 0 || pad_w < 0)
    return 0;
  const int oh = (h + 2 * pad_h - 3) / stride_h + 1, ow = (w + 2 * pad_w - 3) / stride_w + 1;
  if (h + 2 * pad_h < 3 || w + 2 * pad_w < 3 || act_bytes((int64_t)n * h * w, c) > 0x7e000000 || (int64_t)n * oh * ow > INT32_MAX / 2) return 0;
  return (size_t)(c / 32) * (SEP_WAVES / sep_wo(oc / 32)) * 1024 <= SEP_LDS_MOST;
}

int cvmhip_conv2d_separable_i8(const void* xp, const void* wd, const int32_t* bias_d, const cvmhip_chain* chain_d, const void* wp,
                               const int32_t* bias_p, const cvmhip_chain* chain_p, void* out, int n, int c, int h, int w, int oc,
                               int stride_h, int stride_w, int pad_h, int pad_w, void* stream) {
  if (!xp || !wd || !wp || !out || !cvmhip_separable_eligible(n, c, h, w, oc, stride_h, stride_w, pad_h, pad_w) ||
      (((uintptr_t)xp | (uintptr_t)wp | (uintptr_t)out | (uintptr_t)bias_d | (uintptr_t)bias_p) & 15) || ((uintptr_t)wd & 3))
    return arg_error("conv2d_separable_i8");
  SepArgs a = {};
  DevChain cd, cp;
  if (!make_chain(chain_d, &cd) || !make_chain(chain_p, &cp)) return arg_error("conv2d_separable_i8 chain");
  a.first = sep_chain_of(cd);
  a.second = sep_chain_of(cp);
  a.x = reinterpret_cast<const int8_t*>(xp);
  a.wd = reinterpret_cast<const uint32_t*>(wd);
  a.bd = bias_d;
  a.wf = reinterpret_cast<const int8_t*>(wp);
  a.bp = bias_p;
  a.out = reinterpret_cast<int8_t*>(out);
  a.H = h; a.W = w; a.SH = stride_h; a.SW = stride_w; a.PH = pad_h; a.PW = pad_w;
  a.OH = (h + 2 * pad_h - 3) / stride_h + 1;
  a.OW = (w + 2 * pad_w - 3) / stride_w + 1;
  a.P = n * a.OH * a.OW;
  a.ktiles = c / 32;
  a.octiles = oc / 32;
  a.nch1 = (c + 63) / 64 * 2 + 1;
  a.x_bytes = (unsigned)act_bytes((int64_t)n * h * w, c);
  const int wo = sep_wo(a.octiles), wpx = SEP_WAVES / wo;
  a.otgroups = (a.octiles + wo - 1) / wo;
  a.div_ohw = make_fastdiv((uint32_t)(a.OH * a.OW));
  a.div_ow = make_fastdiv((uint32_t)a.OW);
  a.div_groups = make_fastdiv((uint32_t)a.otgroups);
  const int64_t grid = (int64_t)((a.P + 32 * wpx - 1) / (32 * wpx)) * a.otgroups;
  const size_t lds = (size_t)a.ktiles * wpx * 1024;
  char desc[128] = "";
  if (kernel_timing_enabled())
    snprintf(desc, sizeof(desc), "dw 3x3/%d + 1x1 %d->%d in %dx%dx%d out %dx%d tile %dx%d grid %ld", stride_h, c, oc, n, h, w, a.OH, a.OW,
             32 * wo, 32 * wpx, (long)grid);
  KernelTimer timer("k_conv_separable", 2.0 * a.P * c * (9.0 + oc), as_stream(stream),
                    (double)n * h * w * c + (double)c * (9 + oc) + (double)a.P * oc, desc);
  if (wo == 8) k_conv_separable<8><<<(unsigned)grid, 512, lds, as_stream(stream)>>>(a);
  else if (wo == 4) k_conv_separable<4><<<(unsigned)grid, 512, lds, as_stream(stream)>>>(a);
  else if (wo == 2) k_conv_separable<2><<<(unsigned)grid, 512, lds, as_stream(stream)>>>(a);
  else k_conv_separable<1><<<(unsigned)grid, 512, lds, as_stream(stream)>>>(a);
  return check_launch("conv_separable");
}

}  // extern "C"
