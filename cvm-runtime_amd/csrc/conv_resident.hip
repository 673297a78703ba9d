// A run of layers whose maps fit in LDS, one workgroup per image: small networks, and the last layers of larger ones.
//
// What bounds such layers when each is a launch is the launch: an empty kernel and its gap are 1.8 us, the chain of
// prologue, first operands, reduction and drain inside it another 2-3 us, while the arithmetic of a 32 x 32 x 16 layer is a
// few hundred clocks of one compute unit.  Here the activations of an image never leave the compute unit: a layer boundary
// is a workgroup barrier, the filters stream from L2 straight into MFMA operands (the first ones of a layer are requested
// before the barrier in front of it), and the batch spreads over the chip by images.  ResNet-20: 96 us in 23 launches at
// batch 1, 41.5 us in one; 114 us at batch 64, 42.4 us.
//
// Arithmetic: v_mfma_i32_16x16x64_i8 with the filter as the first operand and 16 pixels as the second.  Lane l supplies
// filter row l & 15 and pixel l & 15, both with the 16 bytes (l >> 4) of the 64 bytes of K, and receives channels
// (l >> 4) * 4 .. + 3 of pixel l & 15: four consecutive channels of one pixel, one dword of the result.  (The 32 x 32 form
// of the other kernels would leave half of a 16-channel layer and three quarters of an 8 x 8 map's last tiles empty.)
// LDS layout: NHWC with channels padded to 16 or a multiple of 32 and a border of zeros as wide as the padding of the
// convolutions that read the map: the 16 bytes a lane needs of any tap are one ds_read_b128 at (pixel's place) + (tap's
// place), and 16 neighbouring pixels of a 16-channel map are 256 contiguous bytes.  K is ordered tap by tap; the places of
// the four 16-byte groups of every K step are a table behind the filter.
// What bounds it now (clocks of a 32 x 32 x 16 layer of ResNet-20, 4.2 K in all): 1.5 K of LDS operand reads at 128 bytes a
// clock, about as much of instructions for places and results (2 wavefronts to a SIMD), the rest from barrier to first
// product.  What it took to get there, same network at batch 1: all operand reads of a chunk issued before its first product
// instead of a read and a wait per product, 62 -> 52 us; requests for the first filters inside the loop that uses them, so
// that they land in its registers, 54 -> 45; plain layers in a loop without the tests for the other forms, 45 -> 41.5.  Three
// chunks ahead with four pixel tiles, or 1024 threads, run out of registers (79 us with 28 of them spilled).
#include <string.h>

#include "conv_mfma.h"

namespace cvmhip {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int RES_THREADS = 512, RES_WAVES = RES_THREADS / 64;
constexpr int RES_CHUNK = 3;        // K steps computed together (a 3 x 3 filter over 16, 64, 128, ... channels is whole chunks)
constexpr int RES_HELPERS = 2;     // workgroups per XCD that only touch the filters
constexpr int RES_LDS_MOST = 150 * 1024;

enum { RES_IMAGE = 0, RES_ACT = 1, RES_CONV = 2, RES_SUM = 3, RES_POOL = 4 };
// flags: a chain that is not one clamp and shift; channels past OC exist; the result goes to memory; its map has a border;
// the pixels of every group of tiles exist and lie like the first group's
enum { RES_CHAIN = 1, RES_CHAIN2 = 2, RES_MASK = 4, RES_OUT = 8, RES_BORDER = 16, RES_REGULAR = 32 };

// What the common path of a layer needs, in scalar registers from the layer's first instruction on: read field by field
// where it is used, every field was a trip through the scalar cache in a chain of them.
struct ResHead {
  int kind, tp, items, octiles, chunks, P, OW, flags;
  FastDiv div_ow, div_oct;
  int src, step_y, step_x;          // window of output pixel (0, 0), and bytes to the next row's and column's window
  int dst, dst_row, ocp;            // output pixel (0, 0), bytes of a stored row (dst: -1 = not kept in LDS)
  int res, res_row;                 // residual likewise (res: -1 = none)
  int lo, hi, shift, lo2, hi2, shift2;
  const int8_t* filter;             // [octile][chunk][step][64 lanes][16 bytes]
  const int* taps;                  // [chunk][step][4]: byte offset of the group in the window
  const int32_t* bias;              // octiles * 16 values
  // RES_REGULAR: bytes from a group's first tile to its tile j, in the input, the result and the residual
  int src_off[4], dst_off[4], res_off[4], unused[4];
};
struct __attribute__((aligned(64))) ResLayer {
  ResHead h;
  int C, H, W, cp, map, row;        // IMAGE, ACT: the map; SUM, POOL: the input (map: pixel (0, 0), row: bytes of a stored row)
  int KH, KW, SH, SW, PH, PW, range;
  int OC, out_mode, gcp;            // out_mode: 0 LDS only, 1 int8 act tensor of gcp channels, 2 int32 (image, channel, pixel)
  // border of the output map: start, bytes of a stored row, of the gap between two rows, in front of the first pixel; rows
  int border_at, border_row, border_side, border_edge, border_rows;
  const int8_t* in;                 // IMAGE: int8 NCHW, ACT: act tensor of gcp channels
  void* out;
  DevChain chain, chain2;
};
// the table is read through the scalar cache: nothing in the kernel writes it
typedef const __attribute__((address_space(4))) ResLayer* ResTable;

// Pointers read from the table are generic to the compiler, and a generic access counts as LDS traffic too: every wait for an
// LDS operand would wait for the filter as well.  These say that it is memory.
#define RES_GLOBAL __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ T res_load(const void* p) { return *(const RES_GLOBAL T*)p; }
template <typename T>
__device__ __forceinline__ void res_write(void* p, T v) { *(RES_GLOBAL T*)p = v; }

// (lo <= hi)
__device__ __forceinline__ int res_clamp(int v, int lo, int hi) {
  int r;
  asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "s"(lo), "v"(hi));
  return r;
}

template <typename L>
__device__ __forceinline__ void res_chain(const L& c, int32_t (&v)[4]) {
  const int count = c.count;
#pragma unroll 1
  for (int t = 0; t < count; ++t) {
    const int lo = c.st[t].lo, hi = c.st[t].hi, s1 = c.st[t].s1, add = c.st[t].add, s2 = c.st[t].s2, mul = c.st[t].mul;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = wadd(wmul(res_clamp(v[e], lo, hi), mul) >> s1, add) >> s2;
  }
}

__device__ __forceinline__ uint32_t res_pack(const int32_t (&v)[4]) {
  const uint32_t lo2 = __builtin_amdgcn_perm((uint32_t)v[1], (uint32_t)v[0], 0x0c0c0400u);
  const uint32_t hi2 = __builtin_amdgcn_perm((uint32_t)v[3], (uint32_t)v[2], 0x0c0c0400u);
  return __builtin_amdgcn_perm(hi2, lo2, 0x05040100u);
}

// four channels of pixel p of this image, to LDS byte `at` and wherever else the layer wants them
__device__ __forceinline__ void res_store(const ResHead& h, ResTable L, char* lds, int32_t* out_host, int img, int p, int at, int oc,
                                          const int32_t (&v)[4]) {
  uint32_t d = res_pack(v);
  if (h.flags & RES_MASK) {
    const int left = L->OC - oc;
    d = left >= 4 ? d : left <= 0 ? 0u : d & ((1u << (8 * left)) - 1u);
  }
  if (h.dst >= 0) *reinterpret_cast<uint32_t*>(lds + at) = d;
  if (h.flags & RES_OUT) {
    if (L->out_mode == 1) {
      const int gcp = L->gcp;
      if (oc < gcp) res_write(reinterpret_cast<int8_t*>(L->out) + act_offset((int64_t)img * h.P + p, oc, gcp), d);
    } else {
      const int OC = L->OC;
      const int64_t first = ((int64_t)img * OC + oc) * h.P + p;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (oc + e < OC) {
          res_write(reinterpret_cast<int32_t*>(L->out) + first + (int64_t)e * h.P, v[e]);
          if (out_host) res_write(out_host + first + (int64_t)e * h.P, v[e]);
        }
    }
  }
}

// filter fragments and tap offsets of a chunk
struct ResChunk {
  v4i a[RES_CHUNK];
  int tap[RES_CHUNK];
};
// the chunks an item keeps in flight, and its bias
template <int AHEAD>
struct ResRing {
  ResChunk c[AHEAD];
  v4i bias;
};

// (addresses: a uniform base and the lane's own 32-bit offset)
__device__ __forceinline__ void res_fetch(const ResHead& h, ResChunk& c, int ot, int chunk, int lane) {
  const int8_t* f = h.filter + (unsigned)(ot * h.chunks + chunk) * (RES_CHUNK * 1024u);
  const int8_t* t = reinterpret_cast<const int8_t*>(h.taps) + (unsigned)chunk * (RES_CHUNK * 16u);
#pragma unroll
  for (int u = 0; u < RES_CHUNK; ++u) {
    c.a[u] = res_load<v4i>(f + (unsigned)lane * 16u + u * 1024);
    c.tap[u] = res_load<int>(t + (unsigned)(lane >> 4) * 4u + u * 16);
  }
}

template <int AHEAD>
__device__ __forceinline__ void res_request(const ResHead& h, ResRing<AHEAD>& r, int ot, int lane) {
#pragma unroll
  for (int c = 0; c < AHEAD; ++c)
    if (c < h.chunks) res_fetch(h, r.c[c], ot, c, lane);
  r.bias = res_load<v4i>(reinterpret_cast<const int8_t*>(h.bias) + (unsigned)ot * 64u + (unsigned)(lane >> 4) * 16u);
}

// all operand reads before the first product
template <int TP>
__device__ __forceinline__ void res_chunk(const char* lds, const ResChunk& c, const int (&base)[TP], v4i (&acc)[TP]) {
  v4i x[RES_CHUNK][TP];
#pragma unroll
  for (int u = 0; u < RES_CHUNK; ++u)
#pragma unroll
    for (int j = 0; j < TP; ++j) x[u][j] = *reinterpret_cast<const v4i*>(lds + (base[j] + c.tap[u]));
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < RES_CHUNK; ++u)
#pragma unroll
    for (int j = 0; j < TP; ++j) acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(c.a[u], x[u][j], acc[j], 0, 0, 0);
}

// Byte offsets of lane (l & 15)'s pixel in the input window, the result and the residual.
struct ResPlace {
  int src, dst, res;
};
// pixel p; the channel of the lane's group inside a tile is added where the tile is written
__device__ __forceinline__ ResPlace res_place(const ResHead& h, int p, int lane) {
  const int y = (int)fastdiv((unsigned)p, h.div_ow), x = p - y * h.OW;
  const int column = __mul24(x, h.ocp) + (lane >> 4) * 4;
  ResPlace q;
  q.src = h.src + __mul24(y, h.step_y) + __mul24(x, h.step_x);
  q.dst = h.dst + __mul24(y, h.dst_row) + column;
  q.res = h.res + __mul24(y, h.res_row) + column;
  return q;
}

__device__ __forceinline__ void res_requant(const ResHead& h, const char* lds, int res, int32_t (&v)[4]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = res_clamp(v[e], h.lo, h.hi) >> h.shift;
  if (h.res >= 0) {
    const uint32_t d = *reinterpret_cast<const uint32_t*>(lds + res);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = res_clamp(wadd(v[e], (int32_t)(int8_t)(d >> (8 * e))), h.lo2, h.hi2) >> h.shift2;
  }
}

// A barrier that orders LDS only: requests to memory stay in flight across it (what a layer stores to memory is not read
// inside the launch).
__device__ __forceinline__ void res_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ __forceinline__ void res_border(const ResHead& h, ResTable L, char* lds, int tid) {
  if (h.flags & RES_BORDER) {
    // the border is three runs: in front of the first pixel, behind the last one, and between the rows
    const int row = L->border_row, side = L->border_side, edge = L->border_edge, rows = L->border_rows, at = L->border_at;
    const uint4 zero = make_uint4(0, 0, 0, 0);
    for (int i = tid * 16; i < edge; i += RES_THREADS * 16) {
      *reinterpret_cast<uint4*>(lds + at + i) = zero;
      *reinterpret_cast<uint4*>(lds + at + edge + rows * row - side + i) = zero;
    }
    for (int y = tid; y < rows - 1; y += RES_THREADS)
      for (int i = 0; i < side; i += 16) *reinterpret_cast<uint4*>(lds + at + edge + (y + 1) * row - side + i) = zero;
  }
}

// The first item's operands are requested before the barrier in front of the layer.
// The kernel is bound by instructions (a 16-channel layer has three products per 16 results of a lane group), so the
// regular case keeps everything that does not differ between lanes in scalar registers and knows its tiles' distances.
template <int TP, bool PLAIN>
__device__ __forceinline__ void res_conv(const ResHead& h, ResTable L, char* lds, int32_t* out_host, int img, int wave, int lane) {
  constexpr int AHEAD = TP == 4 ? 2 : 3;   // (four pixel tiles leave registers for two chunks)
  ResRing<AHEAD> r;
  int item = wave, group = (int)fastdiv((unsigned)wave, h.div_oct), ot = wave - group * h.octiles;
  if (item < h.items) res_request(h, r, ot, lane);
  res_barrier();
  res_border(h, L, lds, wave * 64 + lane);
  if (item >= h.items) return;
  const ResPlace own = res_place(h, lane & 15, lane);
  const bool regular = PLAIN || (h.flags & RES_REGULAR);
  for (;;) {
    const int p0 = group * (TP * 16), y0 = (int)fastdiv((unsigned)p0, h.div_ow), x0 = p0 - y0 * h.OW;
    int base[TP];
    if (regular) {
      const int s0 = y0 * h.step_y + x0 * h.step_x;
#pragma unroll
      for (int j = 0; j < TP; ++j) base[j] = own.src + (s0 + h.src_off[j]);
    } else {
#pragma unroll
      for (int j = 0; j < TP; ++j) {
        const int p = p0 + j * 16 + (lane & 15);
        base[j] = res_place(h, p < h.P ? p : 0, lane).src;   // pixels past the map are computed and dropped
      }
    }
    const int oc = ot * 16;
    uint32_t residual[TP];
    if (PLAIN && h.res >= 0) {
      const int r0 = y0 * h.res_row + x0 * h.ocp + oc;
#pragma unroll
      for (int j = 0; j < TP; ++j) residual[j] = *reinterpret_cast<const uint32_t*>(lds + (own.res + (r0 + h.res_off[j])));
    }
    v4i acc[TP];
#pragma unroll
    for (int j = 0; j < TP; ++j) acc[j] = r.bias;
    if (h.chunks <= AHEAD) {
      res_chunk<TP>(lds, r.c[0], base, acc);
      if (h.chunks > 1) res_chunk<TP>(lds, r.c[1], base, acc);
      if (AHEAD > 2 && h.chunks > 2) res_chunk<TP>(lds, r.c[2], base, acc);
    } else {
      // a chunk's registers are requested again, for the chunk AHEAD further on, once it is used
      const int last = h.chunks - 1;
      for (int c = 0;; c += AHEAD) {
        res_chunk<TP>(lds, r.c[0], base, acc);
        if (c == last) break;
        res_fetch(h, r.c[0], ot, min(c + AHEAD, last), lane);
        res_chunk<TP>(lds, r.c[1], base, acc);
        if (c + 1 == last) break;
        res_fetch(h, r.c[1], ot, min(c + AHEAD + 1, last), lane);
        if constexpr (AHEAD > 2) {
          res_chunk<TP>(lds, r.c[2], base, acc);
          if (c + 2 == last) break;
          res_fetch(h, r.c[2], ot, min(c + AHEAD + 2, last), lane);
        }
      }
    }
    if constexpr (PLAIN) {
      const int d0 = y0 * h.dst_row + x0 * h.ocp + oc;
      if (h.res >= 0) {
#pragma unroll
        for (int j = 0; j < TP; ++j) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            acc[j][e] = res_clamp(wadd(res_clamp(acc[j][e], h.lo, h.hi) >> h.shift, (int32_t)(int8_t)(residual[j] >> (8 * e))), h.lo2, h.hi2) >> h.shift2;
        }
      } else {
#pragma unroll
        for (int j = 0; j < TP; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[j][e] = res_clamp(acc[j][e], h.lo, h.hi) >> h.shift;
      }
#pragma unroll
      for (int j = 0; j < TP; ++j) {
        const int32_t v[4] = {acc[j][0], acc[j][1], acc[j][2], acc[j][3]};
        *reinterpret_cast<uint32_t*>(lds + (own.dst + (d0 + h.dst_off[j]))) = res_pack(v);
      }
    } else {
#pragma unroll
      for (int j = 0; j < TP; ++j) {
        const int p = p0 + j * 16 + (lane & 15);
        if (p < h.P) {
          const ResPlace q = res_place(h, p, lane);
          int32_t v[4] = {acc[j][0], acc[j][1], acc[j][2], acc[j][3]};
          if (h.flags & (RES_CHAIN | RES_CHAIN2)) {
            res_chain(L->chain, v);
            if (h.res >= 0) {
              const uint32_t d = *reinterpret_cast<const uint32_t*>(lds + (q.res + oc));
#pragma unroll
              for (int e = 0; e < 4; ++e) v[e] = wadd(v[e], (int32_t)(int8_t)(d >> (8 * e)));
              res_chain(L->chain2, v);
            }
          } else {
            res_requant(h, lds, q.res + oc, v);
          }
          res_store(h, L, lds, out_host, img, p, q.dst + oc, oc + (lane >> 4) * 4, v);
        }
      }
    }
    item += RES_WAVES;
    if (item >= h.items) return;
    const int before = ot;
    group = (int)fastdiv((unsigned)item, h.div_oct);
    ot = item - group * h.octiles;
    if (ot != before || h.chunks > AHEAD) res_request(h, r, ot, lane);   // (else the ring still holds the whole filter)
  }
}

__device__ __forceinline__ ResHead res_head(ResTable L) {
  ResHead h;
  typedef int v16i __attribute__((ext_vector_type(16)));
  static_assert(sizeof(ResHead) == 192, "three lines of the scalar cache");
  const __attribute__((address_space(4))) v16i* w = (const __attribute__((address_space(4))) v16i*)L;
  const v16i part[3] = {w[0], w[1], w[2]};
  __builtin_memcpy(&h, part, sizeof(h));
  return h;
}

__global__ void __launch_bounds__(RES_THREADS) k_conv_resident(const ResLayer* table, int nlayers, int images,
                                                               const cvmhip_resident_call call) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int img = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  ResTable L = (ResTable)table;
  if (img >= images) {
    // Workgroups behind the images: they bring the filters into the L2 of their XCD (workgroups go to the eight XCDs in
    // turn), which the images' workgroups would otherwise wait for layer by layer: every launch starts with an L2 that has
    // to ask memory again, 0.8 us away.
    const int part = (img - ((images + 7) & ~7)) >> 3, parts = ((int)gridDim.x - ((images + 7) & ~7)) >> 3;
    if (img < ((images + 7) & ~7) || (img & 7) >= images) return;
    for (int l = 0; l < nlayers; ++l, ++L) {
      if (L->h.kind != RES_CONV) continue;
      const int8_t* f = L->h.filter;
      const int bytes = L->h.octiles * L->h.chunks * (RES_CHUNK * 1024) + L->h.chunks * (RES_CHUNK * 16);
      int sum = 0;
      for (int at = (part * RES_THREADS + tid) * 128; at < bytes; at += parts * RES_THREADS * 128) sum += res_load<int>(f + at);
      asm volatile("" ::"v"(sum));
    }
    return;
  }
  // The table comes through the scalar cache, which is cold: every wavefront requests an eighth of its lines now, so that a
  // layer does not begin with dependent misses.
  {
    const int lines = nlayers * (int)sizeof(ResLayer) / 64;
    typedef const __attribute__((address_space(4))) int* Word;
    int sum = 0;
    for (int i = wave; i < lines; i += RES_WAVES) sum += *(Word)((uintptr_t)table + 64 * i);
    asm volatile("" ::"s"(sum));
  }
  for (int l = 0; l < nlayers; ++l, ++L) {
    const ResHead h = res_head(L);
    if (h.kind == RES_CONV) {
      const bool plain = (h.flags & (RES_CHAIN | RES_CHAIN2 | RES_MASK | RES_OUT | RES_REGULAR)) == RES_REGULAR;
      if (plain) {
        if (h.tp == 1) res_conv<1, true>(h, L, lds, call.out_host, img, wave, lane);
        else if (h.tp == 2) res_conv<2, true>(h, L, lds, call.out_host, img, wave, lane);
        else res_conv<4, true>(h, L, lds, call.out_host, img, wave, lane);
      } else {
        if (h.tp == 1) res_conv<1, false>(h, L, lds, call.out_host, img, wave, lane);
        else if (h.tp == 2) res_conv<2, false>(h, L, lds, call.out_host, img, wave, lane);
        else res_conv<4, false>(h, L, lds, call.out_host, img, wave, lane);
      }
      continue;
    }
    res_barrier();
    res_border(h, L, lds, tid);
    if (h.kind == RES_IMAGE) {
      const int C = L->C, range = L->range;
      const int8_t* x = (call.image_host ? reinterpret_cast<const int8_t*>(call.image_host) : L->in) + (int64_t)img * C * h.P;
      if (C <= 4 && (h.P & 3) == 0) {
        // four pixels to a thread: all of an image's bytes are requested at once (host memory is 1.5 us away)
        for (int p = tid * 4; p < h.P; p += RES_THREADS * 4) {
          uint32_t d[4];
#pragma unroll
          for (int c = 0; c < 4; ++c) d[c] = res_load<uint32_t>(x + (c < C ? c : C - 1) * h.P + p);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int oy = (int)fastdiv((unsigned)(p + j), h.div_ow), at = h.dst + oy * h.dst_row + (p + j - oy * h.OW) * h.ocp;
            int32_t v[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] = c < C ? res_clamp((int32_t)(int8_t)(d[c] >> (8 * j)), -range, range) : 0;
            *reinterpret_cast<uint4*>(lds + at) = make_uint4(res_pack(v), 0, 0, 0);
            for (int c = 16; c < h.ocp; c += 16) *reinterpret_cast<uint4*>(lds + at + c) = make_uint4(0, 0, 0, 0);
          }
        }
      } else {
        for (int p = tid; p < h.P; p += RES_THREADS) {
          const int oy = (int)fastdiv((unsigned)p, h.div_ow), at = h.dst + oy * h.dst_row + (p - oy * h.OW) * h.ocp;
          for (int c0 = 0; c0 < h.ocp; c0 += 4) {
            int32_t v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = c0 < C ? res_load<int8_t>(x + (int64_t)(c0 + e < C ? c0 + e : C - 1) * h.P + p) : 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = c0 + e < C ? res_clamp(v[e], -range, range) : 0;
            *reinterpret_cast<uint32_t*>(lds + at + c0) = res_pack(v);
          }
        }
      }
    } else if (h.kind == RES_ACT) {
      // granules of 4 bytes: the tensor in memory may have 4 or 8 channels to a pixel
      const int quads = h.ocp >> 2, gcp = L->gcp;
      const int8_t* x = L->in;
      for (int i = tid; i < h.P * quads; i += RES_THREADS) {
        const int p = i / quads, c = (i - p * quads) * 4;
        const int oy = (int)fastdiv((unsigned)p, h.div_ow);
        uint32_t d = 0;
        if (c < gcp) d = res_load<uint32_t>(x + act_offset((int64_t)img * h.P + p, c, gcp));
        *reinterpret_cast<uint32_t*>(lds + h.dst + oy * h.dst_row + (p - oy * h.OW) * h.ocp + c) = d;
      }
    } else if (h.kind == RES_SUM) {
      const int H = L->H, W = L->W, cp = L->cp, map = L->map, row = L->row;
      for (int q = wave; q < (cp >> 2); q += RES_WAVES) {
        int32_t v[4] = {0, 0, 0, 0};
        for (int p = lane; p < H * W; p += 64) {
          const int y = p / W;
          const uint32_t d = *reinterpret_cast<const uint32_t*>(lds + map + y * row + (p - y * W) * cp + q * 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += (int32_t)(int8_t)(d >> (8 * e));
        }
        for (int d = 32; d >= 1; d >>= 1)
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += __shfl_xor(v[e], d, 64);
        res_chain(L->chain, v);
        if (lane == 0) res_store(h, L, lds, call.out_host, img, 0, h.dst + q * 4, q * 4, v);
      }
    } else {
      const int quads = h.ocp >> 2, H = L->H, W = L->W, cp = L->cp, map = L->map, row = L->row;
      const int KH = L->KH, KW = L->KW, SH = L->SH, SW = L->SW, PH = L->PH, PW = L->PW;
      for (int i = tid; i < h.P * quads; i += RES_THREADS) {
        const int p = i / quads, c = (i - p * quads) * 4;
        const int oy = (int)fastdiv((unsigned)p, h.div_ow), ox = p - oy * h.OW;
        int32_t v[4] = {-128, -128, -128, -128};
        for (int r = 0; r < KH; ++r) {
          const int y = oy * SH - PH + r;
          if (y < 0 || y >= H) continue;
          for (int t = 0; t < KW; ++t) {
            const int x = ox * SW - PW + t;
            if (x < 0 || x >= W) continue;
            const uint32_t d = *reinterpret_cast<const uint32_t*>(lds + map + y * row + x * cp + c);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = max(v[e], (int32_t)(int8_t)(d >> (8 * e)));
          }
        }
        res_store(h, L, lds, call.out_host, img, p, h.dst + oy * h.dst_row + ox * h.ocp + c, c, v);
      }
    }
  }
  if (call.flag_host) {
    __threadfence_system();
    __syncthreads();
    if (tid == 0) {
      const uint32_t before = __hip_atomic_fetch_add(call.counter, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
      if (before == (uint32_t)images - 1) {
        *call.counter = 0;
        __hip_atomic_store(call.flag_host, call.ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
  }
}

// int32 OIHW -> fragments (a dword per thread), then the tap table for a map stored with `row` bytes to a row
__global__ void __launch_bounds__(256) k_pack_resident(const int32_t* __restrict__ w, uint32_t* __restrict__ wp, int64_t dwords, int oc,
                                                       int ic, int kh, int kw, int cp, int ksteps, int row, int dh, int dw) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int taps = kh * kw;
  if (i < dwords) {
    const int d = (int)(i & 3), lane = (int)((i >> 2) & 63);
    const int64_t t = i >> 8;
    const int s = (int)(t % ksteps);
    const int64_t o = t / ksteps * 16 + (lane & 15);
    const int k = s * 64 + (lane >> 4) * 16 + d * 4, tap = k / cp, c = k - tap * cp;
    uint32_t pack = 0;
    if (o < oc && tap < taps) {
#pragma unroll
      for (int j = 0; j < 4; ++j) pack |= (c + j < ic ? (uint32_t)(uint8_t)(int8_t)w[((int64_t)o * ic + c + j) * taps + tap] : 0u) << (8 * j);
    }
    wp[i] = pack;
  } else if (i < dwords + ksteps * 4) {
    const int e = (int)(i - dwords), k = e * 16, tap = k / cp, c = k - tap * cp;
    // past the last tap the filter is zero: the window's first bytes will do
    wp[i] = tap < taps ? (uint32_t)((tap / kw) * dh * row + (tap % kw) * dw * cp + c) : 0u;
  }
}

static int res_cp(int c) { return c <= 16 ? 16 : pad_channels(c); }
static int res_chunks(int c, int kh, int kw) { return (kh * kw * res_cp(c) + RES_CHUNK * 64 - 1) / (RES_CHUNK * 64); }
// one clamp and one shift?
static bool res_plain(const DevChain& c, int* lo, int* hi, int* shift) {
  *lo = INT32_MIN;
  *hi = INT32_MAX;
  *shift = 0;
  if (c.count == 0) return true;
  if (c.count > 1 || c.st[0].mul != 1 || c.st[0].add != 0 || (c.st[0].s1 != 0 && c.st[0].s2 != 0)) return false;
  *lo = c.st[0].lo;
  *hi = c.st[0].hi;
  *shift = c.st[0].s1 + c.st[0].s2;
  return true;
}

}  // namespace cvmhip

using namespace cvmhip;

extern "C" {

size_t cvmhip_resident_layer_bytes(void) { return (sizeof(ResLayer) + 63) / 64 * 64; }

size_t cvmhip_resident_lds_limit(void) { return RES_LDS_MOST; }

size_t cvmhip_resident_tensor_bytes(int c, int h, int w, int border_y, int border_x) {
  if (c < 1 || h < 1 || w < 1 || border_y < 0 || border_x < 0 || c > 4096 || h + 2 * border_y > 255 || w + 2 * border_x > 255) return 0;
  return (size_t)res_cp(c) * (h + 2 * border_y) * (w + 2 * border_x);
}

size_t cvmhip_resident_filter_bytes(int oc, int c, int kh, int kw) {
  if (oc < 1 || c < 1 || kh < 1 || kw < 1) return 0;
  return ((size_t)(res_cp(oc) / 16) * 1024 + 16) * res_chunks(c, kh, kw) * RES_CHUNK;
}

int cvmhip_resident_pack_filter(const int32_t* w, void* dst, int oc, int c, int kh, int kw, int dil_h, int dil_w, int stored_w, void* stream) {
  if (!w || !dst || ((uintptr_t)dst & 15) || oc < 1 || c < 1 || c > 4096 || kh < 1 || kw < 1 || dil_h < 1 || dil_w < 1 || stored_w < 1 ||
      stored_w > 255 || (kh - 1) * dil_h > 254 || (kw - 1) * dil_w > 254)
    return arg_error("resident_pack_filter");
  const int ksteps = res_chunks(c, kh, kw) * RES_CHUNK;
  const int64_t dwords = (int64_t)(res_cp(oc) / 16) * ksteps * 256, all = dwords + ksteps * 4;
  k_pack_resident<<<(unsigned)((all + 255) / 256), 256, 0, as_stream(stream)>>>(w, reinterpret_cast<uint32_t*>(dst), dwords, oc, c, kh, kw,
                                                                               res_cp(c), ksteps, stored_w * res_cp(c), dil_h, dil_w);
  return check_launch("resident_pack_filter");
}

int cvmhip_resident_layer(void* table, int index, const cvmhip_resident_desc* d) {
  if (!table || index < 0 || !d) return arg_error("resident_layer");
  auto bytes = [](const cvmhip_resident_map& m) { return cvmhip_resident_tensor_bytes(m.c, m.h, m.w, m.border_y, m.border_x); };
  auto inside = [&](const cvmhip_resident_map& m) {
    return m.at >= 0 && (m.at & 15) == 0 && bytes(m) > 0 && (size_t)m.at + bytes(m) <= RES_LDS_MOST;
  };
  // bytes of a stored row; byte of pixel (y, x)
  auto row = [](const cvmhip_resident_map& m) { return (m.w + 2 * m.border_x) * res_cp(m.c); };
  auto place = [&](const cvmhip_resident_map& m, int y, int x) {
    return m.at + (m.border_y + y) * row(m) + (m.border_x + x) * res_cp(m.c);
  };
  const cvmhip_resident_map &in = d->src, &out = d->dst, &res = d->res;
  const bool load = d->kind == RES_IMAGE || d->kind == RES_ACT;
  ResLayer L = {};
  ResHead& h = L.h;
  h.kind = d->kind;
  if (bytes(out) == 0) return arg_error("resident_layer: map too large");
  h.P = out.h * out.w;
  h.OW = out.w;
  L.OC = out.c;
  h.ocp = res_cp(out.c);
  h.div_ow = make_fastdiv((uint32_t)out.w);
  L.gcp = pad_channels(out.c);
  L.out_mode = d->out_mode;
  L.out = d->out;
  h.flags = (out.c == h.ocp ? 0 : RES_MASK) | (d->out_mode != 0 ? RES_OUT : 0) |
            (out.at >= 0 && (out.border_y > 0 || out.border_x > 0) && !d->border_clean ? RES_BORDER : 0);
  h.dst = h.res = -1;
  if (d->out_mode < 0 || d->out_mode > 2 || (d->out_mode != 0 && !d->out)) return arg_error("resident_layer output");
  if (out.at >= 0) {
    if (!inside(out)) return arg_error("resident_layer output");
    h.dst = place(out, 0, 0);
    h.dst_row = row(out);
    L.border_at = out.at;
    L.border_row = row(out);
    L.border_side = 2 * out.border_x * h.ocp;
    L.border_edge = out.border_y * row(out) + out.border_x * h.ocp;
    L.border_rows = out.h;
  } else if (d->out_mode == 0) {
    return arg_error("resident_layer output");
  }
  if (!make_chain(&d->chain, &L.chain) || !make_chain(&d->chain2, &L.chain2)) return arg_error("resident_layer chain");
  if (!res_plain(L.chain, &h.lo, &h.hi, &h.shift)) h.flags |= RES_CHAIN;
  if (!res_plain(L.chain2, &h.lo2, &h.hi2, &h.shift2)) h.flags |= RES_CHAIN2;
  L.range = d->range;
  if (load) {
    if (!d->in || out.at < 0 || d->out_mode != 0) return arg_error("resident_layer input");
    L.in = reinterpret_cast<const int8_t*>(d->in);
    L.C = out.c; L.H = out.h; L.W = out.w;
  } else {
    if (!inside(in) || d->kh < 1 || d->kw < 1 || d->sh < 1 || d->sw < 1 || d->ph < 0 || d->pw < 0 || d->dh < 1 || d->dw < 1)
      return arg_error("resident_layer operands");
    if (res.at >= 0) {
      if (!inside(res) || res.c != out.c || res.h != out.h || res.w != out.w || d->kind != RES_CONV) return arg_error("resident_layer residual");
      h.res = place(res, 0, 0);
      h.res_row = row(res);
    }
    L.C = in.c; L.H = in.h; L.W = in.w; L.cp = res_cp(in.c);
    L.map = place(in, 0, 0);
    L.row = row(in);
    L.KH = d->kh; L.KW = d->kw; L.SH = d->sh; L.SW = d->sw; L.PH = d->ph; L.PW = d->pw;
    if (d->kind == RES_CONV) {
      if (!d->filter || ((uintptr_t)d->filter & 15) || !d->bias || ((uintptr_t)d->bias & 15)) return arg_error("resident_layer filter");
      // every tap of every window lies inside the stored map
      if (d->ph > in.border_y || d->pw > in.border_x || (out.h - 1) * d->sh - d->ph + (d->kh - 1) * d->dh > in.h - 1 + in.border_y ||
          (out.w - 1) * d->sw - d->pw + (d->kw - 1) * d->dw > in.w - 1 + in.border_x)
        return arg_error("resident_layer window");
      // do all groups of tiles lie alike?
      auto offsets = [&](int tile, int* src_at, int* dst_at, int* res_at) {
        const int y = tile * 16 / out.w, x = tile * 16 % out.w;
        *src_at = y * d->sh * row(in) + x * d->sw * res_cp(in.c);
        *dst_at = y * h.dst_row + x * h.ocp;
        *res_at = y * h.res_row + x * h.ocp;
      };
      h.src = place(in, -d->ph, -d->pw);
      h.step_y = d->sh * row(in);
      h.step_x = d->sw * res_cp(in.c);
      h.chunks = res_chunks(in.c, d->kh, d->kw);
      h.octiles = h.ocp / 16;
      const int ptiles = (h.P + 15) / 16;
      // as many pixel tiles per item (a filter fragment read once serves them all) as still leave every wavefront an item
      h.tp = ptiles * h.octiles >= 4 * RES_WAVES ? 4 : ptiles * h.octiles >= 2 * RES_WAVES ? 2 : 1;
      h.items = h.octiles * ((ptiles + h.tp - 1) / h.tp);
      bool regular = h.P % (16 * h.tp) == 0 && (out.w % 16 == 0 || 16 % out.w == 0);
      for (int t = 0; regular && t < ptiles; ++t) {
        int a[3], b[3];
        offsets(t, &a[0], &a[1], &a[2]);
        offsets(t - t % h.tp, &b[0], &b[1], &b[2]);
        if (t < h.tp) { h.src_off[t] = a[0] - b[0]; h.dst_off[t] = a[1] - b[1]; h.res_off[t] = a[2] - b[2]; }
        else regular = h.src_off[t % h.tp] == a[0] - b[0] && h.dst_off[t % h.tp] == a[1] - b[1] && h.res_off[t % h.tp] == a[2] - b[2];
      }
      if (regular) h.flags |= RES_REGULAR;
      h.div_oct = make_fastdiv((uint32_t)h.octiles);
      h.filter = reinterpret_cast<const int8_t*>(d->filter);
      h.taps = reinterpret_cast<const int*>(h.filter + (size_t)h.octiles * h.chunks * (RES_CHUNK * 1024));
      h.bias = d->bias;
    } else if (d->kind == RES_SUM) {
      if (out.h != 1 || out.w != 1 || in.c != out.c) return arg_error("resident_layer sum");
    } else if (d->kind == RES_POOL) {
      if (in.c != out.c) return arg_error("resident_layer pool");
    } else {
      return arg_error("resident_layer kind");
    }
  }
  memcpy(reinterpret_cast<char*>(table) + index * cvmhip_resident_layer_bytes(), &L, sizeof(L));
  return CVMHIP_OK;
}

int cvmhip_resident_launch(const void* dev_table, int nlayers, int images, size_t lds_bytes, const cvmhip_resident_call* call, double ops,
                           double bytes, void* stream) {
  if (!dev_table || ((uintptr_t)dev_table & 63) || nlayers < 1 || images < 1 || lds_bytes < 16 || lds_bytes > RES_LDS_MOST)
    return arg_error("resident_launch");
  if (call && (!call->image_host || ((uintptr_t)call->image_host & 3) || !call->out_host || !call->counter || !call->flag_host))
    return arg_error("resident_launch call");
  char desc[64] = "";
  if (kernel_timing_enabled()) snprintf(desc, sizeof(desc), "%d layers in LDS, %d images", nlayers, images);
  KernelTimer timer("k_conv_resident", ops, as_stream(stream), bytes, desc);
  const int grid = ((images + 7) & ~7) + 8 * RES_HELPERS;
  k_conv_resident<<<(unsigned)grid, RES_THREADS, lds_bytes, as_stream(stream)>>>(reinterpret_cast<const ResLayer*>(dev_table), nlayers, images,
                                                                                call ? *call : cvmhip_resident_call{});
  return check_launch("conv_resident");
}

}  // extern "C"
