// A run of layers whose maps fit in LDS, one workgroup per image: small networks, and the last layers of larger ones.
//
// What bounds such layers when each is a launch is the launch: an empty kernel and its gap are 1.8 us, the chain of
// prologue, first operands, reduction and drain inside it another 2-3 us, while the arithmetic of a 32 x 32 x 16 layer is a
// few hundred clocks of one compute unit.  Here the activations of an image never leave the compute unit: a layer boundary
// is a workgroup barrier, and the batch spreads over the chip by images.  ResNet-20: 96 us in 23 launches at
// batch 1, 34.4 us in one; 114 us at batch 64, 36 us.
//
// Arithmetic: v_mfma_i32_16x16x64_i8 with the filter as the first operand and 16 pixels as the second.  Lane l supplies
// filter row l & 15 and pixel l & 15, both with the 16 bytes (l >> 4) of the 64 bytes of K, and receives channels
// (l >> 4) * 4 .. + 3 of pixel l & 15: four consecutive channels of one pixel, one dword of the result.  (The 32 x 32 form
// of the other kernels would leave half of a 16-channel layer and three quarters of an 8 x 8 map's last tiles empty.)
// LDS layout: NHWC with channels padded to 16 or a multiple of 32 and a border of zeros as wide as the padding of the
// convolutions that read the map: the 16 bytes a lane needs of any tap are one ds_read_b128 at (pixel's place) + (tap's
// place), and 16 neighbouring pixels of a 16-channel map are 256 contiguous bytes.  K is ordered tap by tap; the places of
// the four 16-byte groups of every K step are a table behind the filter.
// The filter of a layer, its tap offsets, biases and the places of its tiles lie in LDS as well, fetched while the layer in
// front of it is computed.
// What bounds it (ResNet-20, one workgroup; 106 K clocks by the counters when a launch was 39 us): 46 K of LDS transfers, 17 K of them bank
// conflicts, 35 K of vector instructions, 14 K of scalar ones and 13 K of products on each SIMD, which hardly overlap: behind
// a barrier all wavefronts read at the same time and then compute at the same time.  On the way, same network at batch 1:
// all operand reads of a chunk before its first product instead of a read and a wait each 62 -> 52 us; filters requested
// inside the loop that uses them 54 -> 45; plain layers without the tests for other forms 45 -> 41.5; filters and places
// from LDS (no scalar register is spilled any more) and a sum without LDS shuffles 41.5 -> 39; a wavefront beside the others that fetches filters and
// clears borders 39 -> 37, two by two tiles for layers of 32 channels -> 36.5; rows that share operands in layers of 16 -> 34.4.  No difference: 1024 threads, another priority for half of
// the wavefronts, pixels an odd number of granules apart.  Slower: all operands of a 16-channel item of four tiles on their own requested at once, or of a 64-channel one (the
// launch is bound by LDS transfers and vector instructions in turn, not by the latency of either); the next layer's head in scalar registers (spills).
#include <string.h>

#include "conv_mfma.h"
#include "requant.h"

namespace cvmhip {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));

constexpr int RES_THREADS = 512, RES_WAVES = RES_THREADS / 64;   // the wavefronts that compute; one more prepares the next layer
constexpr int RES_CHUNK = 3;        // K steps computed together (a 3 x 3 filter over 16, 64, 128, ... channels is whole chunks)
constexpr int RES_LDS_MOST = 150 * 1024;

enum { RES_IMAGE = 0, RES_ACT = 1, RES_CONV = 2, RES_SUM = 3, RES_POOL = 4 };
// flags: a chain that is not one clamp and shift; channels past OC exist; the result goes to memory; its map has a border;
// none of these, and the pixels of every item exist: the places are in LDS (res_plain_conv)
enum { RES_CHAIN = 1, RES_CHAIN2 = 2, RES_MASK = 4, RES_OUT = 8, RES_BORDER = 16, RES_PLAIN = 32 };

// What the common path of a layer needs, in scalar registers from the layer's first instruction on: read field by field
// where it is used, every field was a trip through the scalar cache in a chain of them.
struct ResHead {
  int kind, tp, items, chunks;
  int flags, w_at, taps_at, bias_at;   // in LDS: fragments [octile][chunk][step][64 lanes][16 bytes], byte offsets in the
                                       // window of the groups [chunk][step][4], biases [octile][16]
  int places_at, residual;             // RES_PLAIN: the lanes' ResPlace, then an ResItem for every item
  int lo, hi, shift, lo2, hi2, shift2;
  // border of the output map: start, bytes of a stored row, of the gap between two rows, in front of the first pixel; rows
  int border_at, border_row, border_side, border_edge, border_rows;
  // filter of the next convolution, to be fetched during this layer: KiB, where to, where from
  int next_kb, next_at, form;           // form: RES_PLAIN: res_form()
  const int8_t* next;
  int unused[6];
};
// Byte offsets of a lane's pixel of a tile, in LDS, without what the tile adds: first tap of the window, result, residual; and
// the lane's bytes of a channel tile's biases.
struct ResPlace {
  int src, dst, res, bias;
};
// What the tiles of an item add to them, and the LDS byte of its filter and of its biases.
struct ResItem {
  int src[4], dst[4], res[4];
  int filter, bias, unused[2];
};
struct __attribute__((aligned(64))) ResLayer {
  ResHead h;
  int octiles, P, OW;
  FastDiv div_ow, div_oct, div_w;
  int src, step_y, step_x;          // window of output pixel (0, 0), and bytes to the next row's and column's window
  int dst, dst_row, ocp;            // output pixel (0, 0), bytes of a stored row (dst: -1 = not kept in LDS)
  int res, res_row;                 // residual likewise (res: -1 = none)
  int C, H, W, cp, map, row;        // IMAGE, ACT: the map; SUM, POOL: the input (map: pixel (0, 0), row: bytes of a stored row)
  int KH, KW, SH, SW, PH, PW, range;
  int OC, out_mode, gcp;            // out_mode: 0 LDS only, 1 int8 act tensor of gcp channels, 2 int32 (image, channel, pixel)
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

// sum over the wavefront, in lane 63: 1, 2, 4 and 8 lanes to the right inside rows of 16, then the rows' last lanes onward
template <int CTRL, int ROWS>
__device__ __forceinline__ int32_t res_add_from(int32_t v) { return v + __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false); }
__device__ __forceinline__ int32_t res_wave_sum(int32_t v) {
  v = res_add_from<0x111, 0xf>(v);
  v = res_add_from<0x112, 0xf>(v);
  v = res_add_from<0x114, 0xf>(v);
  v = res_add_from<0x118, 0xf>(v);
  v = res_add_from<0x142, 0xa>(v);
  return res_add_from<0x143, 0xc>(v);
}

template <typename L>
__device__ __forceinline__ void res_chain(const L& c, int32_t (&v)[4]) {
  const int count = c.count;
#pragma unroll 1
  for (int t = 0; t < count; ++t) {
    const int lo = c.st[t].lo, hi = c.st[t].hi, s1 = c.st[t].s1, add = c.st[t].add, s2 = c.st[t].s2, mul = c.st[t].mul;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = wadd(wmul(clamp_uniform(v[e], lo, hi), mul) >> s1, add) >> s2;
  }
}

// where the pixels of a layer lie, for the forms that are not RES_PLAIN
struct ResGeometry {
  int P, OW;
  FastDiv div_ow;
  int src, step_y, step_x, dst, dst_row, ocp, res, res_row;
};
__device__ __forceinline__ ResGeometry res_geometry(ResTable L) {
  return ResGeometry{L->P, L->OW, FastDiv{L->div_ow.m, L->div_ow.l}, L->src, L->step_y, L->step_x, L->dst, L->dst_row, L->ocp, L->res, L->res_row};
}

// four channels of pixel p of this image, to LDS byte `at` and wherever else the layer wants them
__device__ __forceinline__ void res_store(const ResHead& h, const ResGeometry& q, ResTable L, char* lds, int32_t* out_host, int img, int p, int at, int oc,
                                          const int32_t (&v)[4]) {
  uint32_t d = low_bytes(v[0], v[1], v[2], v[3]);
  if (h.flags & RES_MASK) {
    const int left = L->OC - oc;
    d = left >= 4 ? d : left <= 0 ? 0u : d & ((1u << (8 * left)) - 1u);
  }
  if (q.dst >= 0) *reinterpret_cast<uint32_t*>(lds + at) = d;
  if (h.flags & RES_OUT) {
    if (L->out_mode == 1) {
      const int gcp = L->gcp;
      if (oc < gcp) res_write(reinterpret_cast<int8_t*>(L->out) + act_offset((int64_t)img * q.P + p, oc, gcp), d);
    } else {
      const int OC = L->OC;
      const int64_t first = ((int64_t)img * OC + oc) * q.P + p;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (oc + e < OC) {
          res_write(reinterpret_cast<int32_t*>(L->out) + first + (int64_t)e * q.P, v[e]);
          if (out_host) res_write(out_host + first + (int64_t)e * q.P, v[e]);
        }
    }
  }
}

// A chunk of one item: all operand reads, then the products.  `w`: the lane's bytes of the chunk's first fragment.
template <int TP>
__device__ __forceinline__ void res_chunk(const char* lds, const char* w, const int (&tap)[RES_CHUNK], const int (&base)[TP], v4i (&acc)[TP]) {
  v4i a[RES_CHUNK], x[RES_CHUNK][TP];
#pragma unroll
  for (int u = 0; u < RES_CHUNK; ++u) {
    a[u] = *reinterpret_cast<const v4i*>(w + u * 1024);
#pragma unroll
    for (int j = 0; j < TP; ++j) x[u][j] = *reinterpret_cast<const v4i*>(lds + (base[j] + tap[u]));
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < RES_CHUNK; ++u)
#pragma unroll
    for (int j = 0; j < TP; ++j) acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[u], x[u][j], acc[j], 0, 0, 0);
}

// pixel p; the channel of the lane's group inside a tile is added where the tile is written
__host__ __device__ inline ResPlace res_place(const ResGeometry& g, int p, int y, int lane) {
  const int x = p - y * g.OW, column = x * g.ocp + (lane >> 4) * 4;
  return ResPlace{g.src + y * g.step_y + x * g.step_x, g.dst + y * g.dst_row + column, g.res + y * g.res_row + column, (lane >> 4) * 16};
}

// The end of a layer: its results and the next layer's filter are in LDS.  (The fetches of the filter are not known to the
// compiler, which could not tell them from the operands it waits for.)
__device__ __forceinline__ void res_barrier() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ __forceinline__ void res_fetch_next(const ResHead& h, uint32_t lds_base, int lane) {
  const uint32_t own = (uint32_t)lane * 16u;
  uint32_t to = lds_base + (uint32_t)h.next_at;
  const int8_t* from = h.next;
  int left = h.next_kb;
  // (the s_nop is the wait state between a scalar write to M0 and its use)
  for (; left >= 4; left -= 4, from += 4096, to += 4096)
    asm volatile("s_mov_b32 m0, %5\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %4\n\t"
                 "s_add_u32 m0, %5, 0x400\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %4\n\t"
                 "s_add_u32 m0, %5, 0x800\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %4\n\t"
                 "s_add_u32 m0, %5, 0xc00\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %3, %4" ::"v"(own), "v"(own + 1024u), "v"(own + 2048u), "v"(own + 3072u),
                 "s"(from), "s"(to)
                 : "memory", "scc");
  for (; left > 0; --left, from += 1024, to += 1024)
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(own), "s"(from), "s"(to) : "memory");
}

__device__ __forceinline__ void res_border(const ResHead& h, char* lds, int lane) {
  if (h.flags & RES_BORDER) {
    // the border is three runs: in front of the first pixel, behind the last one, and between the rows
    const int row = h.border_row, side = h.border_side, edge = h.border_edge, rows = h.border_rows, at = h.border_at;
    const uint4 zero = make_uint4(0, 0, 0, 0);
    for (int i = lane * 16; i < edge; i += 64 * 16) {
      *reinterpret_cast<uint4*>(lds + at + i) = zero;
      *reinterpret_cast<uint4*>(lds + at + edge + rows * row - side + i) = zero;
    }
    for (int y = lane; y < rows - 1; y += 64)
      for (int i = 0; i < side; i += 16) *reinterpret_cast<uint4*>(lds + at + edge + (y + 1) * row - side + i) = zero;
  }
}

template <int TP>
__device__ __forceinline__ void res_products(const ResHead& h, const char* lds, const char* w, int lane, int (&tap)[RES_CHUNK],
                                             const int (&base)[TP], v4i (&acc)[TP]) {
  const char* taps = lds + (h.taps_at + (lane >> 4) * 4);
  for (int c = 0; c < h.chunks; ++c) {
    int now[RES_CHUNK];
    const char* after = c + 1 == h.chunks ? taps : taps + (c + 1) * (RES_CHUNK * 16);   // (the next item starts over)
#pragma unroll
    for (int u = 0; u < RES_CHUNK; ++u) {
      now[u] = tap[u];
      tap[u] = *reinterpret_cast<const int*>(after + u * 16);
    }
    res_chunk<TP>(lds, w + c * (RES_CHUNK * 1024), now, base, acc);
  }
  if constexpr (TP == 1) asm volatile(WAIT_8_PASSES : "+v"(acc[0]));
  else if constexpr (TP == 2) asm volatile(WAIT_8_PASSES : "+v"(acc[0]), "+v"(acc[1]));
  else asm volatile(WAIT_8_PASSES : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]));
}
__device__ __forceinline__ void res_first_taps(const ResHead& h, const char* lds, int lane, int (&tap)[RES_CHUNK]) {
#pragma unroll
  for (int u = 0; u < RES_CHUNK; ++u) tap[u] = *reinterpret_cast<const int*>(lds + (h.taps_at + (lane >> 4) * 4 + u * 16));
}

// A convolution with nothing out of the ordinary.  The kernel is bound by instructions (a SIMD issues one in 4 clocks, a
// 16-channel layer has three products per 16 results of a lane group): what differs between the lanes and between the
// items comes from tables that were fetched with the filter, and a layer's own constants fit in scalar registers.
template <int TP>
__device__ __forceinline__ void res_plain_conv(const ResHead& h, char* lds, int wave, int lane) {
  if (wave >= h.items) return;
  const int last = h.residual ? h.shift2 : h.shift;
  const ResPlace own = *reinterpret_cast<const ResPlace*>(lds + (h.places_at + lane * 16));
  const char* rec = lds + (h.places_at + 1024 + wave * 64);
  int tap[RES_CHUNK];
  res_first_taps(h, lds, lane, tap);
  for (int item = wave;;) {
    const v4i src = *reinterpret_cast<const v4i*>(rec), dst = *reinterpret_cast<const v4i*>(rec + 16);
    const int filter = *reinterpret_cast<const int*>(rec + 48), bias_at = *reinterpret_cast<const int*>(rec + 52);
    uint32_t residual[TP];
    if (h.residual) {
      const v4i res = *reinterpret_cast<const v4i*>(rec + 32);
#pragma unroll
      for (int j = 0; j < TP; ++j) residual[j] = *reinterpret_cast<const uint32_t*>(lds + (own.res + res[j]));
    }
    int base[TP];
    v4i acc[TP];
    const v4i bias = *reinterpret_cast<const v4i*>(lds + (bias_at + own.bias));
#pragma unroll
    for (int j = 0; j < TP; ++j) {
      base[j] = own.src + src[j];
      acc[j] = bias;
    }
    res_products<TP>(h, lds, lds + (filter + lane * 16), lane, tap, base, acc);
    if (h.residual) {
#pragma unroll
      for (int j = 0; j < TP; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc[j][e] = clamp_uniform(wadd(clamp_uniform(acc[j][e], h.lo, h.hi) >> h.shift, (int32_t)(int8_t)(residual[j] >> (8 * e))), h.lo2, h.hi2);
      }
    } else {
#pragma unroll
      for (int j = 0; j < TP; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[j][e] = clamp_uniform(acc[j][e], h.lo, h.hi);
    }
#pragma unroll
    for (int j = 0; j < TP; ++j) {
      const int32_t v[4] = {acc[j][0], acc[j][1], acc[j][2], acc[j][3]};
      *reinterpret_cast<uint32_t*>(lds + (own.dst + dst[j])) = shift_to_bytes(v[0], v[1], v[2], v[3], last);
    }
    item += RES_WAVES;
    if (item >= h.items) return;
    rec += RES_WAVES * 64;
  }
}

// The same for layers of an even number of channel tiles and STEPS of K known here: TM channel tiles share the operands of TP pixel
// tiles, all of an item's operands are requested at once, and the next item's behind its products.  Two by two tiles take a
// 16 x 16 x 32 layer from 2 600 to 2 330 clocks (3 050 to 2 660 with a residual) against one by four.
template <int TM, int TP, int STEPS>
__device__ __forceinline__ void res_item_conv(const ResHead& h, char* lds, int wave, int lane) {
  if (wave >= h.items) return;
  const int last = h.residual ? h.shift2 : h.shift;
  const ResPlace own = *reinterpret_cast<const ResPlace*>(lds + (h.places_at + lane * 16));
  const char* rec = lds + (h.places_at + 1024 + wave * 64);
  int tap[STEPS];
#pragma unroll
  for (int u = 0; u < STEPS; ++u) tap[u] = *reinterpret_cast<const int*>(lds + (h.taps_at + (lane >> 4) * 4 + u * 16));
  const int next_channels = h.chunks * (RES_CHUNK * 1024);   // from a channel tile's filter to the next one's
  v4i a[STEPS][TM], x[STEPS][TP], acc[TM][TP], bias[TM], src, dst, res;
  uint32_t residual[TM][TP];
  int filter, bias_at;
  auto record = [&]() {
    src = *reinterpret_cast<const v4i*>(rec);
    filter = *reinterpret_cast<const int*>(rec + 48);
    bias_at = *reinterpret_cast<const int*>(rec + 52);
    dst = *reinterpret_cast<const v4i*>(rec + 16);
    if (h.residual) res = *reinterpret_cast<const v4i*>(rec + 32);
  };
  auto request = [&]() {
#pragma unroll
    for (int u = 0; u < STEPS; ++u) {
#pragma unroll
      for (int m = 0; m < TM; ++m) a[u][m] = *reinterpret_cast<const v4i*>(lds + (filter + lane * 16) + m * next_channels + u * 1024);
#pragma unroll
      for (int j = 0; j < TP; ++j) x[u][j] = *reinterpret_cast<const v4i*>(lds + (own.src + src[j] + tap[u]));
    }
  };
  record();
  request();
  for (int item = wave;;) {
    const v4i to = dst, beside = res;
#pragma unroll
    for (int m = 0; m < TM; ++m) {
      bias[m] = *reinterpret_cast<const v4i*>(lds + (bias_at + own.bias + m * 64));
      if (h.residual) {
#pragma unroll
        for (int j = 0; j < TP; ++j) residual[m][j] = *reinterpret_cast<const uint32_t*>(lds + (own.res + beside[j] + m * 16));
      }
    }
    item += RES_WAVES;
    const bool more = item < h.items;
    if (more) {
      rec += RES_WAVES * 64;
      record();
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int j = 0; j < TP; ++j) acc[m][j] = bias[m];
#pragma unroll
    for (int u = 0; u < STEPS; ++u)
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int j = 0; j < TP; ++j) acc[m][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[u][m], x[u][j], acc[m][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    if (more) request();
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int j = 0; j < TP; ++j) asm volatile(WAIT_8_PASSES : "+v"(acc[m][j]));
    if (h.residual) {
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int j = 0; j < TP; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            acc[m][j][e] = clamp_uniform(wadd(clamp_uniform(acc[m][j][e], h.lo, h.hi) >> h.shift, (int32_t)(int8_t)(residual[m][j] >> (8 * e))), h.lo2, h.hi2);
    } else {
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int j = 0; j < TP; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[m][j][e] = clamp_uniform(acc[m][j][e], h.lo, h.hi);
    }
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int j = 0; j < TP; ++j) {
        const int32_t v[4] = {acc[m][j][0], acc[m][j][1], acc[m][j][2], acc[m][j][3]};
        *reinterpret_cast<uint32_t*>(lds + (own.dst + to[j] + m * 16)) = shift_to_bytes(v[0], v[1], v[2], v[3], last);
      }
    if (!more) return;
  }
}
// 3 x 3 over 16 channels, stride 1: K is ordered (column of the window, row), four rows to a step with a filter of zeros for the fourth
// (res_pair_order), so the operand that one output row reads holds the rows of the output row below it as well: the same
// operand times the filter moved on by one row of the window.  Six operands serve four tiles where res_plain_conv reads
// twelve, the filter stays in registers, and an item's operands are requested behind the products of the one in front of it;
// tiles 2 and 3 of an item lie below tiles 0 and 1.  A 32 x 32 x 16 layer: 3 550 -> 2 970 clocks, 4 300 -> 3 560 with a residual
// (of these 770 products, and 1 000 or 1 800 vector instructions of each SIMD's four items).
__device__ __forceinline__ void res_pair_conv(const ResHead& h, char* lds, int wave, int lane) {
  if (wave >= h.items) return;
  const int last = h.residual ? h.shift2 : h.shift;
  const int group = lane >> 4;
  const char* rec = lds + (h.places_at + 1024 + wave * 64);
  struct Record {   // of an ResItem
    v2i src, at;    // at: filter, bias
    v4i dst, res;
  } now, next;
  auto record = [&](Record& r) {
    r.src = *reinterpret_cast<const v2i*>(rec);
    r.at = *reinterpret_cast<const v2i*>(rec + 48);
    r.dst = *reinterpret_cast<const v4i*>(rec + 16);
    r.res = *reinterpret_cast<const v4i*>(rec + 32);
    rec += RES_WAVES * 64;
  };
  // all that has a known place, then all that these say, so that a layer begins with two waits for LDS
  const ResPlace own = *reinterpret_cast<const ResPlace*>(lds + (h.places_at + lane * 16));
  record(now);
  int tap[3];
#pragma unroll
  for (int u = 0; u < 3; ++u) tap[u] = *reinterpret_cast<const int*>(lds + (h.taps_at + u * 16 + min(group, 2) * 4));
  const int row1 = *reinterpret_cast<const int*>(lds + (h.taps_at + 4)), row2 = *reinterpret_cast<const int*>(lds + (h.taps_at + 8));
  int item = wave + RES_WAVES;
  if (item < h.items) record(next);
  __builtin_amdgcn_sched_barrier(0);
  const int below = group == 3 ? row2 - row1 : 0;   // (the table's fourth row is no row)
#pragma unroll
  for (int u = 0; u < 3; ++u) tap[u] += own.src + below;
  v4i a[2][3], x[3][2], bias;
  uint32_t residual[4];
  int loaded = -1;
  auto request = [&](const Record& r) {
#pragma unroll
    for (int u = 0; u < 3; ++u)
#pragma unroll
      for (int j = 0; j < 2; ++j) x[u][j] = *reinterpret_cast<const v4i*>(lds + (r.src[j] + tap[u]));
    const int at = __builtin_amdgcn_readfirstlane(r.at[0]);
    if (at != loaded) {
      loaded = at;
#pragma unroll
      for (int u = 0; u < 3; ++u) {
        a[0][u] = *reinterpret_cast<const v4i*>(lds + (at + u * 1024 + lane * 16));
        a[1][u] = *reinterpret_cast<const v4i*>(lds + (at + u * 1024 + (group ? lane - 16 : 48 + lane) * 16));   // (a step's last 16 lanes hold zeros)
      }
    }
    bias = *reinterpret_cast<const v4i*>(lds + (r.at[1] + own.bias));
  };
  auto beside = [&](const Record& r) {
    if (h.residual) {
#pragma unroll
      for (int j = 0; j < 4; ++j) residual[j] = *reinterpret_cast<const uint32_t*>(lds + (own.res + r.res[j]));
    }
  };
  request(now);
  beside(now);
  for (;;) {
    const bool more = item < h.items;
    const v4i to = now.dst;
    __builtin_amdgcn_sched_barrier(0);
    v4i acc[4] = {bias, bias, bias, bias};
#pragma unroll
    for (int u = 0; u < 3; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[j >> 1][u], x[u][j & 1], acc[j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    if (more) request(next);
    asm volatile(WAIT_8_PASSES : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]));
    if (h.residual) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc[j][e] = clamp_uniform(wadd(clamp_uniform(acc[j][e], h.lo, h.hi) >> h.shift, (int32_t)(int8_t)(residual[j] >> (8 * e))), h.lo2, h.hi2);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[j][e] = clamp_uniform(acc[j][e], h.lo, h.hi);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int32_t v[4] = {acc[j][0], acc[j][1], acc[j][2], acc[j][3]};
      *reinterpret_cast<uint32_t*>(lds + (own.dst + to[j])) = shift_to_bytes(v[0], v[1], v[2], v[3], last);
    }
    if (!more) return;
    beside(next);
    now = next;
    item += RES_WAVES;
    if (item < h.items) record(next);
  }
}
constexpr int RES_PAIR = 1;   // ResHead::form
// does the filter of a layer have the order (column, row) of res_pair_conv?  (All layers that could have it do: the places of its
// groups come from a table, any kernel takes them.)
__host__ __device__ constexpr bool res_pair_order(int kh, int kw, int cp) { return kh == 3 && kw == 3 && cp == 16; }

// (TM, TP, STEPS) of res_item_conv in one number; 0: res_plain_conv
__host__ __device__ constexpr int res_form(int tm, int tp, int steps) { return steps * 16 + tm * 8 - 8 + tp; }
#define RES_FORMS(F) F(2, 2, 3) F(2, 2, 5)

// any convolution, one pixel tile at a time
__device__ __forceinline__ void res_conv(const ResHead& h, ResTable L, char* lds, int32_t* out_host, int img, int wave, int lane) {
  const ResGeometry g = res_geometry(L);
  const FastDiv div_oct{L->div_oct.m, L->div_oct.l};
  const int octiles = L->octiles;
  int tap[RES_CHUNK];
  res_first_taps(h, lds, lane, tap);
  for (int item = wave; item < h.items; item += RES_WAVES) {
    const int group = (int)fastdiv((unsigned)item, div_oct), ot = item - group * octiles, oc = ot * 16;
    const int pixel = group * 16 + (lane & 15), p = pixel < g.P ? pixel : 0;   // pixels past the map are computed and dropped
    const ResPlace q = res_place(g, p, (int)fastdiv((unsigned)p, g.div_ow), lane);
    const int base[1] = {q.src};
    v4i acc[1] = {*reinterpret_cast<const v4i*>(lds + (h.bias_at + ot * 64 + q.bias))};
    res_products<1>(h, lds, lds + (h.w_at + ot * h.chunks * (RES_CHUNK * 1024) + lane * 16), lane, tap, base, acc);
    if (pixel >= g.P) continue;
    int32_t v[4] = {acc[0][0], acc[0][1], acc[0][2], acc[0][3]};
    const bool chains = h.flags & (RES_CHAIN | RES_CHAIN2);
    if (chains) {
      res_chain(L->chain, v);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = clamp_uniform(v[e], h.lo, h.hi) >> h.shift;
    }
    if (h.residual) {
      const uint32_t d = *reinterpret_cast<const uint32_t*>(lds + (q.res + oc));
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = wadd(v[e], (int32_t)(int8_t)(d >> (8 * e)));
      if (chains) {
        res_chain(L->chain2, v);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = clamp_uniform(v[e], h.lo2, h.hi2) >> h.shift2;
      }
    }
    res_store(h, g, L, lds, out_host, img, pixel, q.dst + oc, oc + (lane >> 4) * 4, v);
  }
}

__device__ __forceinline__ ResHead res_head(ResTable L) {
  ResHead h;
  typedef int v16i __attribute__((ext_vector_type(16)));
  static_assert(sizeof(ResHead) == 128, "two lines of the scalar cache");
  const __attribute__((address_space(4))) v16i* w = (const __attribute__((address_space(4))) v16i*)L;
  const v16i part[2] = {w[0], w[1]};
  __builtin_memcpy(&h, part, sizeof(h));
  return h;
}

__global__ void __launch_bounds__(RES_THREADS + 64) k_conv_resident(const ResLayer* table, int nlayers, int images,
                                                               const cvmhip_resident_call call) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int img = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  ResTable L = (ResTable)table;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  // The table comes through the scalar cache, which is cold: every wavefront requests an eighth of its lines now, so that a
  // layer does not begin with dependent misses.
  {
    const int lines = nlayers * (int)sizeof(ResLayer) / 64;
    typedef const __attribute__((address_space(4))) int* Word;
    int sum = 0;
    for (int i = wave; i < lines; i += RES_WAVES + 1) sum += *(Word)((uintptr_t)table + 64 * i);
    asm volatile("" ::"s"(sum));
  }
  // The last wavefront fetches the next layer's filter and clears the border of this layer's map while the others compute: as
  // the first thing all of them did behind the barrier it was 300 to 1 600 of a layer's 4 000 clocks.
  if (wave == RES_WAVES) {
    for (int l = 0; l < nlayers; ++l, ++L) {
      const ResHead h = res_head(L);
      res_barrier();
      res_fetch_next(h, lds_base, lane);
      res_border(h, lds, lane);
    }
  } else {
  for (int l = 0; l < nlayers; ++l, ++L) {
    const ResHead h = res_head(L);
    res_barrier();
    if (h.flags & RES_PLAIN) {
#define RES_CASE(TM, TP, STEPS) case res_form(TM, TP, STEPS): res_item_conv<TM, TP, STEPS>(h, lds, wave, lane); continue;
      switch (h.form) {
        RES_FORMS(RES_CASE)
        case RES_PAIR: res_pair_conv(h, lds, wave, lane); continue;
        default: break;
      }
#undef RES_CASE
      if (h.tp == 1) res_plain_conv<1>(h, lds, wave, lane);
      else if (h.tp == 2) res_plain_conv<2>(h, lds, wave, lane);
      else res_plain_conv<4>(h, lds, wave, lane);
      continue;
    }
    if (h.kind == RES_CONV) {
      res_conv(h, L, lds, call.out_host, img, wave, lane);
      continue;
    }
    const ResGeometry g = res_geometry(L);
    if (h.kind == RES_IMAGE) {
      const int C = L->C, range = L->range;
      const int8_t* x = (call.image_host ? reinterpret_cast<const int8_t*>(call.image_host) : L->in) + (int64_t)img * C * g.P;
      if (C <= 4 && (g.P & 3) == 0) {
        // four pixels to a thread: all of an image's bytes are requested at once (host memory is 1.5 us away)
        for (int p = tid * 4; p < g.P; p += RES_THREADS * 4) {
          uint32_t d[4];
#pragma unroll
          for (int c = 0; c < 4; ++c) d[c] = res_load<uint32_t>(x + (c < C ? c : C - 1) * g.P + p);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int oy = (int)fastdiv((unsigned)(p + j), g.div_ow), at = g.dst + oy * g.dst_row + (p + j - oy * g.OW) * g.ocp;
            int32_t v[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] = c < C ? clamp_uniform((int32_t)(int8_t)(d[c] >> (8 * j)), -range, range) : 0;
            *reinterpret_cast<uint4*>(lds + at) = make_uint4(low_bytes(v[0], v[1], v[2], v[3]), 0, 0, 0);
            for (int c = 16; c < g.ocp; c += 16) *reinterpret_cast<uint4*>(lds + at + c) = make_uint4(0, 0, 0, 0);
          }
        }
      } else {
        for (int p = tid; p < g.P; p += RES_THREADS) {
          const int oy = (int)fastdiv((unsigned)p, g.div_ow), at = g.dst + oy * g.dst_row + (p - oy * g.OW) * g.ocp;
          for (int c0 = 0; c0 < g.ocp; c0 += 4) {
            int32_t v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = c0 < C ? res_load<int8_t>(x + (int64_t)(c0 + e < C ? c0 + e : C - 1) * g.P + p) : 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = c0 + e < C ? clamp_uniform(v[e], -range, range) : 0;
            *reinterpret_cast<uint32_t*>(lds + at + c0) = low_bytes(v[0], v[1], v[2], v[3]);
          }
        }
      }
    } else if (h.kind == RES_ACT) {
      // granules of 4 bytes: the tensor in memory may have 4 or 8 channels to a pixel
      const int quads = g.ocp >> 2, gcp = L->gcp;
      const int8_t* x = L->in;
      for (int i = tid; i < g.P * quads; i += RES_THREADS) {
        const int p = i / quads, c = (i - p * quads) * 4;
        const int oy = (int)fastdiv((unsigned)p, g.div_ow);
        uint32_t d = 0;
        if (c < gcp) d = res_load<uint32_t>(x + act_offset((int64_t)img * g.P + p, c, gcp));
        *reinterpret_cast<uint32_t*>(lds + g.dst + oy * g.dst_row + (p - oy * g.OW) * g.ocp + c) = d;
      }
    } else if (h.kind == RES_SUM) {
      const int H = L->H, W = L->W, cp = L->cp, map = L->map, row = L->row;
      const FastDiv div_w{L->div_w.m, L->div_w.l};
      for (int q = wave; q < (cp >> 2); q += RES_WAVES) {
        int32_t v[4] = {0, 0, 0, 0};
        for (int p = lane; p < H * W; p += 64) {
          const int y = (int)fastdiv((unsigned)p, div_w);
          const uint32_t d = *reinterpret_cast<const uint32_t*>(lds + map + y * row + (p - y * W) * cp + q * 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += (int32_t)(int8_t)(d >> (8 * e));
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = res_wave_sum(v[e]);
        res_chain(L->chain, v);
        if (lane == 63) res_store(h, g, L, lds, call.out_host, img, 0, g.dst + q * 4, q * 4, v);
      }
    } else {
      const int quads = g.ocp >> 2, H = L->H, W = L->W, cp = L->cp, map = L->map, row = L->row;
      const int KH = L->KH, KW = L->KW, SH = L->SH, SW = L->SW, PH = L->PH, PW = L->PW;
      for (int i = tid; i < g.P * quads; i += RES_THREADS) {
        const int p = i / quads, c = (i - p * quads) * 4;
        const int oy = (int)fastdiv((unsigned)p, g.div_ow), ox = p - oy * g.OW;
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
        res_store(h, g, L, lds, call.out_host, img, p, g.dst + oy * g.dst_row + ox * g.ocp + c, c, v);
      }
    }
  }
  }
  if (call.flag_host) {
    const uint32_t ticket = tid == 0 ? call.counter[1] + 1 : 0;
    stores_done_barrier();
    if (tid == 0) {
      __threadfence_system();
      const uint32_t before = __hip_atomic_fetch_add(call.counter, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
      if (before == (uint32_t)images - 1) {
        call.counter[0] = 0;
        call.counter[1] = ticket;
        __hip_atomic_store(call.flag_host, ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
  }
}

// int32 OIHW -> fragments (a dword per thread), then the tap table for a map stored with `row` bytes to a row, then the bias
__global__ void __launch_bounds__(256) k_pack_resident(const int32_t* __restrict__ w, const int32_t* __restrict__ bias, uint32_t* __restrict__ wp,
                                                       int64_t dwords, int octiles, int oc,
                                                       int ic, int kh, int kw, int cp, int ksteps, int row, int dh, int dw) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int taps = kh * kw;
  if (i < dwords) {
    const int d = (int)(i & 3), lane = (int)((i >> 2) & 63);
    const int64_t t = i >> 8;
    const int s = (int)(t % ksteps);
    const int64_t o = t / ksteps * 16 + (lane & 15);
    const bool pair = res_pair_order(kh, kw, cp);
    const int k = s * 64 + (lane >> 4) * 16 + d * 4;
    const int tap = pair ? (lane >> 4 < 3 && s < 3 ? (lane >> 4) * 3 + s : taps) : k / cp, c = pair ? d * 4 : k - tap * cp;
    uint32_t pack = 0;
    if (o < oc && tap < taps) {
#pragma unroll
      for (int j = 0; j < 4; ++j) pack |= (c + j < ic ? (uint32_t)(uint8_t)(int8_t)w[((int64_t)o * ic + c + j) * taps + tap] : 0u) << (8 * j);
    }
    wp[i] = pack;
  } else if (i < dwords + ksteps * 4) {
    const int e = (int)(i - dwords), k = e * 16;
    const bool pair = res_pair_order(kh, kw, cp);
    const int tap = pair ? (e % 4 < 3 && e < 12 ? e % 4 * 3 + e / 4 : taps) : k / cp, c = pair ? 0 : k - tap * cp;
    // past the last tap the filter is zero: the window's first bytes will do
    wp[i] = tap < taps ? (uint32_t)((tap / kw) * dh * row + (tap % kw) * dw * cp + c) : 0u;
  } else if (i < dwords + ksteps * 4 + octiles * 16) {
    const int o = (int)(i - dwords - ksteps * 4);
    wp[i] = bias && o < oc ? (uint32_t)bias[o] : 0u;
  }
}

static int res_cp(int c) { return c <= 16 ? 16 : pad_channels(c); }
static int res_chunks(int c, int kh, int kw) { return (kh * kw * res_cp(c) + RES_CHUNK * 64 - 1) / (RES_CHUNK * 64); }

}  // namespace cvmhip

using namespace cvmhip;

extern "C" {

size_t cvmhip_resident_layer_bytes(void) { return (sizeof(ResLayer) + 63) / 64 * 64; }

size_t cvmhip_resident_lds_limit(void) { return RES_LDS_MOST; }

size_t cvmhip_resident_tensor_bytes(int c, int h, int w, int border_y, int border_x) {
  if (c < 1 || h < 1 || w < 1 || border_y < 0 || border_x < 0 || c > 4096 || h + 2 * border_y > 255 || w + 2 * border_x > 255) return 0;
  return (size_t)res_cp(c) * (h + 2 * border_y) * (w + 2 * border_x);
}

// Tiles of an item, as many as still leave every wavefront one: a filter fragment read once serves all pixel tiles, an activation
// operand all channel tiles.  Two by two reads 8 operands for 8 products of two steps where one by four reads 10.
struct ResTiling {
  int tm, tp, form;
};
static ResTiling res_tiling(int ptiles, int octiles, int steps) {
  const int tp = ptiles * octiles >= 4 * RES_WAVES ? 4 : ptiles * octiles >= 2 * RES_WAVES ? 2 : 1;
  auto known = [&](int tm, int t) {
#define RES_KNOWN(TM, TP, STEPS) if (tm == TM && t == TP && steps == STEPS) return true;
    RES_FORMS(RES_KNOWN)
#undef RES_KNOWN
    return false;
  };
  if (tp == 4 && octiles % 2 == 0 && ptiles % 2 == 0 && known(2, 2)) return {2, 2, res_form(2, 2, steps)};
  return {1, tp, 0};
}
static int res_steps(int c, int kh, int kw) { return (kh * kw * res_cp(c) + 63) / 64; }
static size_t res_places_at(int oc, int c, int kh, int kw) {
  return ((size_t)(res_cp(oc) / 16) * 1024 + 16) * res_chunks(c, kh, kw) * RES_CHUNK + (size_t)res_cp(oc) * 4;
}

size_t cvmhip_resident_filter_bytes(int oc, int c, int kh, int kw, int oh, int ow) {
  if (oc < 1 || c < 1 || kh < 1 || kw < 1 || oh < 1 || ow < 1) return 0;
  const int ptiles = (oh * ow + 15) / 16, octiles = res_cp(oc) / 16;
  const ResTiling t = res_tiling(ptiles, octiles, res_steps(c, kh, kw));
  return (res_places_at(oc, c, kh, kw) + 1024 + (size_t)(octiles / t.tm) * ((ptiles + t.tp - 1) / t.tp) * sizeof(ResItem) + 1023) / 1024 * 1024;
}

int cvmhip_resident_pack_filter(const int32_t* w, const int32_t* bias, void* dst, int oc, int c, int kh, int kw, int dil_h, int dil_w,
                                int stored_w, void* stream) {
  if (!w || !dst || ((uintptr_t)dst & 15) || oc < 1 || c < 1 || c > 4096 || kh < 1 || kw < 1 || dil_h < 1 || dil_w < 1 || stored_w < 1 ||
      stored_w > 255 || (kh - 1) * dil_h > 254 || (kw - 1) * dil_w > 254)
    return arg_error("resident_pack_filter");
  const int ksteps = res_chunks(c, kh, kw) * RES_CHUNK;
  const int64_t dwords = (int64_t)(res_cp(oc) / 16) * ksteps * 256, all = dwords + ksteps * 4 + res_cp(oc);
  k_pack_resident<<<(unsigned)((all + 255) / 256), 256, 0, as_stream(stream)>>>(w, bias, reinterpret_cast<uint32_t*>(dst), dwords,
                                                                               res_cp(oc) / 16, oc, c, kh, kw, res_cp(c), ksteps,
                                                                               stored_w * res_cp(c), dil_h, dil_w);
  return check_launch("resident_pack_filter");
}

int cvmhip_resident_layer(void* table, int index, const cvmhip_resident_desc* d, void* places, size_t* places_bytes, size_t* places_off) {
  if (!table || index < 0 || !d || !places || !places_bytes || !places_off) return arg_error("resident_layer");
  *places_bytes = *places_off = 0;
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
  L.P = out.h * out.w;
  L.OW = out.w;
  L.OC = out.c;
  L.ocp = res_cp(out.c);
  L.div_ow = make_fastdiv((uint32_t)out.w);
  L.gcp = pad_channels(out.c);
  L.out_mode = d->out_mode;
  L.out = d->out;
  h.flags = (out.c == L.ocp ? 0 : RES_MASK) | (d->out_mode != 0 ? RES_OUT : 0) |
            (out.at >= 0 && (out.border_y > 0 || out.border_x > 0) && !d->border_clean ? RES_BORDER : 0);
  L.dst = L.res = -1;
  if (d->out_mode < 0 || d->out_mode > 2 || (d->out_mode != 0 && !d->out)) return arg_error("resident_layer output");
  if (out.at >= 0) {
    if (!inside(out)) return arg_error("resident_layer output");
    L.dst = place(out, 0, 0);
    L.dst_row = row(out);
    h.border_at = out.at;
    h.border_row = row(out);
    h.border_side = 2 * out.border_x * L.ocp;
    h.border_edge = out.border_y * row(out) + out.border_x * L.ocp;
    h.border_rows = out.h;
  } else if (d->out_mode == 0) {
    return arg_error("resident_layer output");
  }
  if (!make_chain(&d->chain, &L.chain) || !make_chain(&d->chain2, &L.chain2)) return arg_error("resident_layer chain");
  if (!clamp_shift_of(L.chain, &h.lo, &h.hi, &h.shift)) h.flags |= RES_CHAIN;
  if (!clamp_shift_of(L.chain2, &h.lo2, &h.hi2, &h.shift2)) h.flags |= RES_CHAIN2;
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
      L.res = place(res, 0, 0);
      L.res_row = row(res);
      h.residual = 1;
    }
    L.C = in.c; L.H = in.h; L.W = in.w; L.cp = res_cp(in.c);
    L.map = place(in, 0, 0);
    L.row = row(in);
    L.KH = d->kh; L.KW = d->kw; L.SH = d->sh; L.SW = d->sw; L.PH = d->ph; L.PW = d->pw;
    if (d->kind == RES_CONV) {
      const size_t blob = cvmhip_resident_filter_bytes(out.c, in.c, d->kh, d->kw, out.h, out.w);
      if (!d->filter || ((uintptr_t)d->filter & 15) || d->filter_at < 0 || (d->filter_at & 15) || d->filter_at + blob > RES_LDS_MOST || index < 1)
        return arg_error("resident_layer filter");
      // every tap of every window lies inside the stored map
      if (d->ph > in.border_y || d->pw > in.border_x || (out.h - 1) * d->sh - d->ph + (d->kh - 1) * d->dh > in.h - 1 + in.border_y ||
          (out.w - 1) * d->sw - d->pw + (d->kw - 1) * d->dw > in.w - 1 + in.border_x)
        return arg_error("resident_layer window");
      L.src = place(in, -d->ph, -d->pw);
      L.step_y = d->sh * row(in);
      L.step_x = d->sw * res_cp(in.c);
      L.octiles = L.ocp / 16;
      L.div_oct = make_fastdiv((uint32_t)L.octiles);
      h.chunks = res_chunks(in.c, d->kh, d->kw);
      h.w_at = d->filter_at;
      h.taps_at = h.w_at + L.octiles * h.chunks * (RES_CHUNK * 1024);
      h.bias_at = h.taps_at + h.chunks * (RES_CHUNK * 16);
      // whole tiles, which all lie like the first one (part of a row, or whole rows), and a result for LDS only
      const int ptiles = (L.P + 15) / 16;
      const ResTiling tiling = res_tiling(ptiles, L.octiles, res_steps(in.c, d->kh, d->kw));
      const int tp = tiling.tp, groups = L.octiles / tiling.tm;
      const bool narrow = h.residual ? clamp_shift_narrow(h.lo2, h.hi2, h.shift2) : clamp_shift_narrow(h.lo, h.hi, h.shift);
      if (narrow && !(h.flags & (RES_CHAIN | RES_CHAIN2 | RES_MASK | RES_OUT)) && L.P % (16 * tp) == 0 && (out.w % 16 == 0 || 16 % out.w == 0)) {
        h.flags |= RES_PLAIN;
        h.tp = tp;
        h.form = tiling.form;
        h.items = groups * (ptiles / tp);
        // tiles one above the other: two of a row and the two below them, or four of a map one tile wide
        const bool pair = res_pair_order(d->kh, d->kw, res_cp(in.c)) && d->sh == 1 && d->sw == 1 && d->dh == 1 && d->dw == 1 && tp == 4 && tiling.tm == 1 &&
                          (out.w % 32 == 0 ? out.h % 2 == 0 : out.w == 16 && out.h % 4 == 0);
        if (pair) h.form = RES_PAIR;
        const size_t at = res_places_at(out.c, in.c, d->kh, d->kw);
        h.places_at = h.w_at + (int)at;
        const ResGeometry g = {L.P, L.OW, L.div_ow, L.src, L.step_y, L.step_x, L.dst, L.dst_row, L.ocp, L.res, L.res_row};
        ResPlace* own = reinterpret_cast<ResPlace*>(places);
        ResItem* items = reinterpret_cast<ResItem*>(own + 64);
        for (int l = 0; l < 64; ++l) own[l] = res_place(g, l & 15, (l & 15) / g.OW, l);
        const ResPlace first = res_place(g, 0, 0, 0);
        for (int i = 0; i < h.items; ++i) {
          const int ot = i % groups * tiling.tm;
          items[i] = ResItem{};
          items[i].filter = h.w_at + ot * h.chunks * (RES_CHUNK * 1024);
          items[i].bias = h.bias_at + ot * 64;
          for (int t = 0; t < tp; ++t) {
            int p = (i / groups * tp + t) * 16;
            if (pair && out.w == 16) {
              p = i / groups * 64 + ((t & 1) * 2 + (t >> 1)) * 16;
            } else if (pair) {
              const int across = out.w / 32, g2 = i / groups, y = g2 / across * 2 + (t >> 1), x = (g2 % across) * 32 + (t & 1) * 16;
              p = y * out.w + x;
            }
            const ResPlace q = res_place(g, p, p / g.OW, 0);
            items[i].src[t] = q.src - first.src;
            items[i].dst[t] = q.dst - first.dst + ot * 16;
            items[i].res[t] = q.res - first.res + ot * 16;
          }
        }
        *places_off = at;
        *places_bytes = 64 * sizeof(ResPlace) + h.items * sizeof(ResItem);
      } else {
        h.items = L.octiles * ptiles;
      }
      // the layer in front of it fetches the filter
      ResHead before;
      char* at = reinterpret_cast<char*>(table) + (index - 1) * cvmhip_resident_layer_bytes();
      memcpy(&before, at, sizeof(before));
      before.next = reinterpret_cast<const int8_t*>(d->filter);
      before.next_kb = (int)(blob / 1024);
      before.next_at = d->filter_at;
      memcpy(at, &before, sizeof(before));
    } else if (d->kind == RES_SUM) {
      L.div_w = make_fastdiv((uint32_t)in.w);
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
  k_conv_resident<<<(unsigned)images, RES_THREADS + 64, lds_bytes, as_stream(stream)>>>(reinterpret_cast<const ResLayer*>(dev_table), nlayers, images,
                                                                                  call ? *call : cvmhip_resident_call{});
  return check_launch("conv_resident");
}

}  // extern "C"
