// conv2d on int32 tensors in one launch: both operands are read as the caller holds them (NCHW and OIHW, int32), narrowed in
// registers and multiplied by the matrix cores.
//
// The general path packs both operands to int8 fragments first and then multiplies: two launches and, for every value, four
// bytes read and one written before the product reads it again.  A plug-in host calls such a layer once per node, so the
// launches are most of it at one image and the extra pass a third of it at sixteen.
//
// Lane l of v_mfma_i32_32x32x32_i8 supplies 16 values of K for row l & 31 of an operand.  K is dealt so that lanes 0..31 take the first half
// of the input channels and lanes 32..63 the second: what differs between the halves is then one constant per operand.  K is ordered
// (channel, tap), as the filter lies in memory: a lane's 16 filter values are 64 contiguous bytes; its 16 activation values are 16
// requests, each 2 x 32 neighbouring pixels, at offsets that are the same for all lanes (a table of 16 per phase of the taps, in
// the kernel's arguments).  A tap outside the image is a bit per pixel and tap, masked after the packing.
#include "conv_mfma.h"

namespace cvmhip {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

struct DirectArgs {
  const int32_t *x, *w, *bias;
  int32_t* y;
  int C, first, HW, K;          // input channels, those of lanes 0..31; input pixels of a channel; C * taps
  int half, chunks, whole;      // values of K in lanes 0..31; chunks of 16 of them; the chunks in which every lane has 16
  int OC, OHW, OW, P, octiles, H, W, SH, SW, PH, PW, DH, DW;
  unsigned x_bytes;
  FastDiv div_ohw, div_ow;
  int tab[9][16];               // byte offset of value j behind the first channel of a chunk that begins at tap `phase`
};

// four values of K to a dword
__device__ __forceinline__ int direct_pack(int a, int b, int c, int d) {
  const uint32_t lo = __builtin_amdgcn_perm((uint32_t)b, (uint32_t)a, 0x0c0c0400u), hi = __builtin_amdgcn_perm((uint32_t)d, (uint32_t)c, 0x0c0c0400u);
  return (int)__builtin_amdgcn_perm(hi, lo, 0x05040100u);
}

// a pixel of the output: byte offset of its window's first tap in this half's channels, taps inside the image (three times over, so
// that a shift by a chunk's phase gives 16), element of its first output channel
struct DirectPixel {
  unsigned off, valid, out;
};
template <int TAPS, bool MASK>
__device__ __forceinline__ DirectPixel direct_pixel(const DirectArgs& a, int p0, int h) {
  const int p = p0 < a.P ? p0 : a.P - 1;
  const int img = (int)fastdiv((unsigned)p, a.div_ohw), pix = p - img * a.OHW;
  const int oy = (int)fastdiv((unsigned)pix, a.div_ow), iy = oy * a.SH - a.PH, ix = (pix - oy * a.OW) * a.SW - a.PW;
  DirectPixel q = {(unsigned)(((img * a.C + h * a.first) * a.HW + iy * a.W + ix) * 4), 0, (unsigned)(img * a.OC * a.OHW + pix)};
  if constexpr (MASK) {
#pragma unroll
    for (int t = 0; t < TAPS; ++t) {
      const int r = TAPS == 1 ? 0 : t / 3, s = TAPS == 1 ? 0 : t % 3;
      if ((unsigned)(iy + r * a.DH) < (unsigned)a.H && (unsigned)(ix + s * a.DW) < (unsigned)a.W) q.valid |= 1u << t;
    }
    q.valid = TAPS == 1 ? (q.valid ? 0xffffu : 0u) : q.valid | q.valid << 9 | q.valid << 18;
  }
  return q;
}
// A lane's 16 activation values of chunk c.  An offset past the tensor, or in front of it, gives zero: the range is checked on the sum.
template <int TAPS>
__device__ __forceinline__ void direct_request(const DirectArgs& a, __amdgpu_buffer_rsrc_t xs, unsigned off, int c, int (&v)[16]) {
  const int channel = TAPS == 1 ? c * 16 : (c * 16) / 9, phase = TAPS == 1 ? 0 : c * 16 - channel * 9;
  const int* tab = a.tab[phase];
  const unsigned base = off + (unsigned)(channel * a.HW * 4);
#pragma unroll
  for (int j = 0; j < 16; ++j) v[j] = (int)__builtin_amdgcn_raw_buffer_load_b32(xs, (int)(base + (unsigned)tab[j]), 0, 0);
}
template <int TAPS, bool MASK>
__device__ __forceinline__ v4i direct_fragment(const int (&v)[16], unsigned valid, int c) {
  const unsigned in = TAPS == 1 ? valid : valid >> (c * 16 - (c * 16) / 9 * 9);
  v4i f;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    int d = direct_pack(v[g * 4], v[g * 4 + 1], v[g * 4 + 2], v[g * 4 + 3]);
    if constexpr (MASK) d &= (int)((__umul24((in >> (g * 4)) & 15u, 0x204081u) & 0x1010101u) * 255u);   // four bits to four bytes of ones
    f[g] = d;
  }
  return f;
}

// Few tiles: a workgroup computes 32 output channels x 32 pixels, its eight wavefronts an eighth of K each.
// Bound by the requests of a chunk (the four of the filter touch 64 lines each), 300 clocks a compute unit.
constexpr int DIRECT_SPLIT = 8;
template <int TAPS, bool MASK>
__global__ void __launch_bounds__(DIRECT_SPLIT * 64) k_conv_direct(const DirectArgs a) {
  __shared__ int s_part[DIRECT_SPLIT * 16 * 64];
  const int lane = threadIdx.x & 63, col = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // the tiles of one range of pixels run on one XCD: they share its activations in the L2
  const int xcd = blockIdx.x & 7, per = gridDim.x >> 3, extra = gridDim.x & 7;
  const int pid = xcd * per + (xcd < extra ? xcd : extra) + (blockIdx.x >> 3);
  const int tile = pid / a.octiles, oc0 = (pid - tile * a.octiles) * 32, px = tile * 32 + col;
  const __amdgpu_buffer_rsrc_t xs = __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(a.x), 0, (int)a.x_bytes, 0x00020000);
  const DirectPixel q = direct_pixel<TAPS, MASK>(a, px, h);
  const int here = h ? a.K - a.half : a.half;   // values of K this lane has (0: one input channel)
  const int32_t* row = a.w + (int64_t)(oc0 + col < a.OC ? oc0 + col : a.OC - 1) * a.K + (here ? h * a.half : 0);
  // two registers of the tile are added up and stored by each wavefront
  int sum[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int reg = wave * 2 + i, oc = oc0 + 8 * (reg >> 2) + 4 * h + (reg & 3);
    sum[i] = a.bias ? a.bias[oc < a.OC ? oc : a.OC - 1] : 0;
  }

  const int c_begin = a.chunks * wave / DIRECT_SPLIT, c_end = a.chunks * (wave + 1) / DIRECT_SPLIT;
  typedef int v4u __attribute__((ext_vector_type(4), aligned(4)));   // rows need not start on 16 bytes
  struct Fetch {
    v4i f[4];
    int v[16];
  };
  auto request = [&](int c, Fetch& t) {
    direct_request<TAPS>(a, xs, q.off, c, t.v);
    if (c < a.whole) {
#pragma unroll
      for (int g = 0; g < 4; ++g) t.f[g] = *reinterpret_cast<const v4u*>(row + c * 16 + g * 4);
    } else {
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int k = c * 16 + j, f = row[k < here ? k : 0];
        t.f[j >> 2][j & 3] = k < here ? f : 0;
      }
    }
  };
  v16i acc = {};
  auto multiply = [&](int c, const Fetch& t) {
    v4i f;
#pragma unroll
    for (int g = 0; g < 4; ++g) f[g] = direct_pack(t.f[g][0], t.f[g][1], t.f[g][2], t.f[g][3]);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(f, direct_fragment<TAPS, MASK>(t.v, q.valid, c), acc, 0, 0, 0);
  };
  Fetch t[2];
  if (c_begin < c_end) request(c_begin, t[0]);
  int c = c_begin;
  for (; c + 2 <= c_end; c += 2) {
    request(c + 1, t[1]);
    multiply(c, t[0]);
    if (c + 2 < c_end) request(c + 2, t[0]);
    multiply(c + 1, t[1]);
  }
  if (c < c_end) multiply(c, t[0]);
#pragma unroll
  for (int i = 0; i < 16; ++i) s_part[(wave * 16 + i) * 64 + lane] = acc[i];
  __syncthreads();
#pragma unroll
  for (int s = 0; s < DIRECT_SPLIT; ++s)
#pragma unroll
    for (int i = 0; i < 2; ++i) sum[i] = wadd(sum[i], s_part[(s * 16 + wave * 2 + i) * 64 + lane]);
  if (px >= a.P) return;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int reg = wave * 2 + i, oc = oc0 + 8 * (reg >> 2) + 4 * h + (reg & 3);
    if (oc < a.OC) a.y[q.out + (unsigned)(oc * a.OHW)] = sum[i];
  }
}

// More tiles than the chip has places: a workgroup packs the filter rows of 32 * TM output channels into LDS once and then takes one
// group of 128 pixels after another, 32 to a wavefront, with D chunks of activations in flight across the groups.
// Bound by the int32 tensors (16 x 256 x 56 x 56 to 64 channels: 15.0 us for 64 MB) and by the chain in front of the first product: filter, packing, barrier.
// Filter rows of 96 to 256 channels a workgroup: 20 to 150 % slower (fewer wavefronts wait for more).
template <int TAPS, bool MASK, int TM, int D>
__global__ void __launch_bounds__(256) k_conv_slab(const DirectArgs a) {
  extern __shared__ __attribute__((aligned(16))) v4i s_filter[];   // [m][chunk][lane]
  const int lane = threadIdx.x & 63, col = lane & 31, h = lane >> 5, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int xcd = blockIdx.x & 7, per = gridDim.x >> 3, extra = gridDim.x & 7;
  const int pid = xcd * per + (xcd < extra ? xcd : extra) + (blockIdx.x >> 3), stride = gridDim.x / a.octiles;
  int group = pid / a.octiles;
  const int oc0 = (pid - group * a.octiles) * (32 * TM), groups = (a.P + 127) >> 7, own = wave * 32 + col;
  const __amdgpu_buffer_rsrc_t xs = __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(a.x), 0, (int)a.x_bytes, 0x00020000);
  DirectPixel now = direct_pixel<TAPS, MASK>(a, group * 128 + own, h), ahead = now;
  int v[D][16], ahead_group = group, ahead_c = 0;
  auto request = [&](int (&q)[16]) {   // the next chunk of the sequence
    if (ahead_group >= groups) return;
    direct_request<TAPS>(a, xs, ahead.off, ahead_c, q);
    if (++ahead_c == a.chunks) {
      ahead_c = 0;
      ahead_group += stride;
      if (ahead_group < groups) ahead = direct_pixel<TAPS, MASK>(a, ahead_group * 128 + own, h);
    }
  };
#pragma unroll
  for (int d = 0; d < D; ++d) request(v[d]);

  typedef int v4u __attribute__((ext_vector_type(4), aligned(4)));
  // a thread packs four values at a time: four threads a lane's 64 bytes, sixteen lanes to a request, eight requests in flight
  {
    constexpr int BATCH = 8 / TM;
    const int l = threadIdx.x >> 2, g = threadIdx.x & 3, half = l >> 5, here = half ? a.K - a.half : a.half;
    const int32_t* row[TM];
#pragma unroll
    for (int m = 0; m < TM; ++m) {
      const int oc = oc0 + m * 32 + (l & 31);
      row[m] = a.w + (int64_t)(oc < a.OC ? oc : a.OC - 1) * a.K + (here ? half * a.half : 0);
    }
    for (int c0 = 0; c0 < a.chunks; c0 += BATCH) {
      v4u f[TM][BATCH];
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
          const int k = (c0 + u) * 16 + g * 4;
          f[m][u] = *reinterpret_cast<const v4u*>(k + 4 <= here ? row[m] + k : a.w);
        }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
          const int k = (c0 + u) * 16 + g * 4;
          if (c0 + u >= a.chunks) continue;
          int d = k + 4 <= here ? direct_pack(f[m][u][0], f[m][u][1], f[m][u][2], f[m][u][3]) : 0;
          if (k < here && k + 4 > here)   // the end of a half that is not whole quads
            d = direct_pack(row[m][k], k + 1 < here ? row[m][k + 1] : 0, k + 2 < here ? row[m][k + 2] : 0, 0);
          reinterpret_cast<int*>(s_filter)[((m * a.chunks + c0 + u) * 64 + l) * 4 + g] = d;
        }
    }
  }
  int bias[TM][16];
  v16i acc[TM];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int oc = oc0 + m * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
      acc[m][i] = bias[m][i] = a.bias ? a.bias[oc < a.OC ? oc : a.OC - 1] : 0;
    }
  __syncthreads();
  for (int c = 0;;) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const v4i f = direct_fragment<TAPS, MASK>(v[d], now.valid, c);
      request(v[d]);
#pragma unroll
      for (int m = 0; m < TM; ++m) acc[m] = __builtin_amdgcn_mfma_i32_32x32x32_i8(s_filter[(m * a.chunks + c) * 64 + lane], f, acc[m], 0, 0, 0);
      if (++c == a.chunks) {
        if (group * 128 + own < a.P) {
#pragma unroll
          for (int m = 0; m < TM; ++m)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              const int oc = oc0 + m * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
              if (oc < a.OC) a.y[now.out + (unsigned)(oc * a.OHW)] = acc[m][i];
            }
        }
        group += stride;
        if (group >= groups) return;
        now = direct_pixel<TAPS, MASK>(a, group * 128 + own, h);
        c = 0;
#pragma unroll
        for (int m = 0; m < TM; ++m)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[m][i] = bias[m][i];
      }
    }
  }
}

// Which layers, us here against packing and product (the launch that is saved is 2-3 us of host time on top).  All figures on these kernels are us of a layer in a
// replayed graph, with four sets of operands in turn where nothing else is said.
// 1 x 1, k_conv_direct up to 448 tiles of 32 x 32 and K of 640: 256 -> 64 at 56 x 56 4.2 / 6.9, two images of it (392 tiles) 5.6 / 7.9, four
// (784) 8.9 / 9.8; 512 -> 128 at 28 x 28 5.3 / 6.5; K = 1024 9.5 / 7.0.  k_conv_slab beyond that up to K = 256: 64 -> 256 at 56 x 56 4.5 / 7.0,
// 16 images 16.5 / 19.0; 256 -> 64, four images 7.1 / 9.8, 16 15.0 / 20.4; 96 -> 160 at 4 x 75 x 75 9.5 / 13.3; 256 -> 320 at 8 x 96 x 96 53.0 / 52.5; 256 -> 1024 at
// 16 x 14 x 14 12.4 / 11.7, 256 -> 256 at 8 x 28 x 28 9.2 / 9.4; K = 512 at 4 x 28 x 28 9.6 / 7.9, 16 images 13.8 / 13.2.
// 3 x 3, k_conv_direct up to 256 tiles and K of 640: 64 -> 64 at 56 x 56 5.7 / 7.0; two images (392 tiles) 8.2 / 7.2; K = 1152 at 28 x 28 7.9 / 8.3.
constexpr int DIRECT_TILES = 448, DIRECT_TILES_3X3 = 256, DIRECT_K = 640, SLAB_K = 256, SLAB_GROUPS = 512;

// The chip holds two workgroups of k_conv_slab to a compute unit at once; more take their groups in rounds (one round of 528 took 11.7 where two of 264 take 10.5).
static int64_t slab_rounds(int64_t groups, int oc, int tm) { return (groups * ((oc + 32 * tm - 1) / (32 * tm)) + SLAB_GROUPS - 1) / SLAB_GROUPS; }

// 32 channels to a workgroup, not 64, where these are no more rounds (one: more wavefronts share the wait; more: less of the last 64 channels is past the layer's end).
// us with 64 and 32, two chunks in flight (workgroups); here and below with four sets of operands in turn | with sets of 700 MB:
//   64 -> 256 at 56 x 56 (100, 200) 5.4 4.5, 200 -> 64 at 96 x 96 (72, 144) 8.9 7.1, 96 -> 160 at 2 x 75 x 75 (264, 440) 7.4 6.5 | 8.4 8.1, 128 -> 64 at 6 x 75 x 75 (264, 528) 9.7 10.3;
//   96 -> 160 at 4 x 75 x 75 (528, 880) 10.6 9.8 | 12.4 12.0, 128 -> 96 at 5 x 91 x 91 (648, 972) 12.7 11.1; a round more: 107 -> 269 at 5 x 59 x 59 (680, 1224) 12.9 13.4, 184 -> 205 at 3 x 87 x 87 (712,
//   1246) 15.2 16.2, 96 -> 160 at 6 x 75 x 75 (792, 1320) 11.9 11.6 | 15.0 16.3, 64 -> 64 at 12 x 75 x 75 (528, 1056) 11.7 10.6 | 14.1 14.8; but with few channels, half of the last 64 past the end and
//   two rounds half empty 48 -> 200 at 5 x 70 x 70 (768, 1344) 10.8 10.1 | 12.7 12.2, 46 -> 202 at 6 x 59 x 59 (656, 1148) 10.9 10.2 | 12.5 12.1, 80 -> 224 at 9 x 48 x 48 (648, 1134) 11.0 10.6
static bool slab_narrow(int64_t groups, int ic, int oc) {
  const int64_t wide = groups * ((oc + 63) / 64);
  const bool half = oc % 64 > 0 && oc % 64 <= 32 && wide > SLAB_GROUPS && wide <= 800 && ic <= 80;
  return slab_rounds(groups, oc, 1) <= slab_rounds(groups, oc, 2) + (half ? 1 : 0);
}

// Four chunks of activations in flight, not two (six: as four).  us with two and four, by how many workgroups there are and how many of them read the same pixels:
//   at most one to a compute unit: 256 -> 64 at 4 x 56 x 56 (196) 8.1 7.2 | 11.8 8.2, 200 -> 64 at 96 x 96 (144) 7.1 6.2
//   one round, one to its pixels: 128 -> 64 at 9 x 75 x 75 (396) 10.6 11.4 | 13.5 14.6, 200 -> 64 at 7 x 75 x 75 (308) 12.5 13.4 | 16.1 17.3, 256 -> 64 at 12 x 56 x 56 (294) 12.8 13.6 | 16.3 16.8;
//     only 256 -> 64 at 16 x 56 x 56 (392) 15.0 15.0 | 18.4 17.9, at 20 (490) | 20.2 19.7
//   one round, several: 256 -> 128 at 8 x 56 x 56 (392) | 15.4 15.0, 240 -> 182 at 77 x 77 (282) 8.8 9.0 | 10.8 10.0, 194 -> 133 at 7 x 52 x 52 (444) | 13.4 12.8; few channels 128 -> 64 at
//     5 x 75 x 75 (440) 7.8 8.1, 96 -> 160 at 2 x 75 x 75 (440) 6.5 6.7 | 8.1 8.3, 77 -> 156 at 2 x 94 x 94 (417) 8.4 8.8 | 10.0 10.3
//   rounds, one or two: 128 -> 64 at 12 x 75 x 75 (528) 13.9 14.9 | 19.8 20.0, 256 -> 64 at 24 x 56 x 56 (588) 25.9 27.4 | 25.9 27.4, 200 -> 64 at 16 x 91 x 91 (1036) 40.1 41.2 | 40.2 41.3;
//     96 -> 64 at 12 x 96 x 96 (864) 17.8 16.9 | 18.6 18.2, 64 -> 128 at 10 x 96 x 96 (1440) 20.4 18.6 | 19.7 18.9, 128 -> 96 at 10 x 91 x 91 (1294) 24.0 24.3 | 23.3 23.8
//   rounds, three or more: 233 -> 214 at 5 x 88 x 88 (1212) 28.9 24.9, 148 -> 277 at 8 x 64 x 64 (1280) 18.0 16.5, 64 -> 256 at 16 x 56 x 56 (1568) 19.6 17.2 | 22.7 20.8
static bool slab_deep(int64_t workgroups, int octiles, int chunks) {
  if (workgroups <= SLAB_GROUPS / 2) return true;
  if (octiles >= 3) return workgroups > SLAB_GROUPS || chunks >= 5;
  if (octiles == 2) return workgroups > 800 || chunks >= 5;
  return workgroups > 800 ? chunks <= 4 : workgroups > 320 && workgroups <= SLAB_GROUPS && chunks >= 8;
}

static bool conv_direct(const int32_t* x, const int32_t* w, const int32_t* bias, int32_t* y, int n, int ic, int h, int wd, int oc, int oh, int ow, int kh,
                 int kw, int stride_h, int stride_w, int pad_h, int pad_w, int dil_h, int dil_w, hipStream_t s, int* rc) {
  const bool one = kh == 1 && kw == 1;
  if (!one && !(kh == 3 && kw == 3)) return false;
  const int64_t pixels = (int64_t)n * oh * ow, bytes = (int64_t)n * ic * h * wd * 4, filter = (int64_t)oc * ic * kh * kw;
  if (filter < 4 || bytes > INT32_MAX || filter > INT32_MAX / 4 || pixels * oc > INT32_MAX || pixels > INT32_MAX - 4096) return false;
  // what a tap's offset adds to a pixel's stays inside 31 bits, on either side of the tensor
  if ((int64_t)(16 + 2 * dil_h + pad_h) * h * wd * 4 + (int64_t)(2 * dil_w + pad_w + 1) * 4 + bytes > INT32_MAX) return false;
  const bool mask = pad_h > 0 || pad_w > 0;
  const int64_t tiles = (pixels + 31) / 32 * ((oc + 31) / 32);
  const int K = ic * kh * kw;
  const bool few = tiles <= (one ? DIRECT_TILES : DIRECT_TILES_3X3) && K <= DIRECT_K;
  if (!few && !(one && K <= SLAB_K)) return false;
  DirectArgs a = {};
  a.x = x; a.w = w; a.bias = bias; a.y = y;
  const int taps = kh * kw;
  a.C = ic;
  a.first = (ic + 1) / 2;
  a.HW = h * wd;
  a.K = ic * taps;
  a.half = a.first * taps;
  a.chunks = (a.half + 15) / 16;
  a.whole = (a.K - a.half) / 16;
  a.OC = oc; a.OHW = oh * ow; a.OW = ow; a.P = (int)pixels;
  a.H = h; a.W = wd; a.SH = stride_h; a.SW = stride_w; a.PH = pad_h; a.PW = pad_w; a.DH = dil_h; a.DW = dil_w;
  a.x_bytes = (unsigned)bytes;
  a.div_ohw = make_fastdiv((uint32_t)a.OHW);
  a.div_ow = make_fastdiv((uint32_t)ow);
  for (int p = 0; p < (one ? 1 : 9); ++p)
    for (int j = 0; j < 16; ++j) {
      const int c = one ? j : (p + j) / 9, t = one ? 0 : (p + j) % 9;
      a.tab[p][j] = (c * a.HW + (t / 3) * dil_h * wd + (t % 3) * dil_w) * 4;
    }
  char desc[128] = "";
  if (kernel_timing_enabled())
    snprintf(desc, sizeof(desc), "%dx%d/%d %d->%d in %dx%dx%d out %dx%d i32 operands, i32 out", kh, kw, stride_h, ic, oc, n, h, wd, oh, ow);
  KernelTimer timer(few ? "k_conv_direct" : "k_conv_slab", 2.0 * (double)pixels * oc * K, s, (double)bytes + 4.0 * (double)filter + 4.0 * (double)pixels * oc, desc);
  if (few) {
    a.octiles = (oc + 31) / 32;
    const unsigned blocks = (unsigned)tiles;
    if (one && !mask) k_conv_direct<1, false><<<blocks, DIRECT_SPLIT * 64, 0, s>>>(a);
    else if (one) k_conv_direct<1, true><<<blocks, DIRECT_SPLIT * 64, 0, s>>>(a);
    else if (mask) k_conv_direct<9, true><<<blocks, DIRECT_SPLIT * 64, 0, s>>>(a);
    else k_conv_direct<9, false><<<blocks, DIRECT_SPLIT * 64, 0, s>>>(a);
  } else {
    const int64_t groups = (pixels + 127) / 128;
    const int tm = slab_narrow(groups, ic, oc) ? 1 : 2;
    a.octiles = (oc + 32 * tm - 1) / (32 * tm);
    const int64_t rounds = slab_rounds(groups, oc, tm);
    const bool deep = slab_deep(groups * a.octiles, a.octiles, a.chunks);
    const unsigned blocks = (unsigned)((groups + rounds - 1) / rounds * a.octiles);
    const size_t lds = (size_t)tm * a.chunks * 1024;
#define SLAB_CASE(MASK, TM, D) k_conv_slab<1, MASK, TM, D><<<blocks, 256, lds, s>>>(a)
    if (mask) {
      if (tm == 1) { if (deep) SLAB_CASE(true, 1, 4); else SLAB_CASE(true, 1, 2); }
      else if (deep) SLAB_CASE(true, 2, 4);
      else SLAB_CASE(true, 2, 2);
    } else if (tm == 1) { if (deep) SLAB_CASE(false, 1, 4); else SLAB_CASE(false, 1, 2); }
    else if (deep) SLAB_CASE(false, 2, 4);
    else SLAB_CASE(false, 2, 2);
#undef SLAB_CASE
  }
  *rc = check_launch("conv_direct");
  return true;
}

}  // namespace cvmhip

using namespace cvmhip;

extern "C" {

int cvmhip_conv2d(const int32_t* x, const int32_t* w, const int32_t* bias, int32_t* y,
                  int n, int ic, int h, int wd, int oc, int kh, int kw,
                  int stride_h, int stride_w, int pad_h, int pad_w, int dil_h, int dil_w,
                  int groups, void* workspace, size_t workspace_bytes, void* stream) {
  if (!x || !w || !y) return arg_error("conv2d null tensor");
  if (n < 1 || ic < 1 || h < 1 || wd < 1 || oc < 1 || kh < 1 || kw < 1 || stride_h < 1 || stride_w < 1 ||
      pad_h < 0 || pad_w < 0 || dil_h < 1 || dil_w < 1 || groups < 1 || ic % groups || oc % groups)
    return arg_error("conv2d attributes");
  const int oh = (h + 2 * pad_h - (dil_h * (kh - 1) + 1)) / stride_h + 1;
  const int ow = (wd + 2 * pad_w - (dil_w * (kw - 1) + 1)) / stride_w + 1;
  if (h + 2 * pad_h < dil_h * (kh - 1) + 1 || wd + 2 * pad_w < dil_w * (kw - 1) + 1) return arg_error("conv2d kernel exceeds input");
  hipStream_t s = as_stream(stream);
  if (groups > 1)
    return conv_grouped_i32(x, w, bias, y, n, ic, h, wd, oc, oh, ow, kh, kw, stride_h, stride_w, pad_h, pad_w, dil_h, dil_w, groups, s);
  const size_t need = cvmhip_conv2d_workspace_bytes(n, ic, h, wd, oc, kh, kw, 1);
  if (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 255)) return arg_error("conv2d workspace");
  int rc;
  if (!conv_kernel_forced() && conv_direct(x, w, bias, y, n, ic, h, wd, oc, oh, ow, kh, kw, stride_h, stride_w, pad_h, pad_w, dil_h, dil_w, s, &rc))
    return rc;
  return conv2d_two_launches(x, w, bias, y, n, ic, h, wd, oc, oh, ow, kh, kw, stride_h, stride_w, pad_h, pad_w, dil_h, dil_w, workspace, s);
}

}  // extern "C"
