// The way of an int8 image batch into the row-window layout of the first convolution (conv_mfma.h: StemGeom), straight from
// pinned host memory and while the host is still copying the caller's bytes there.
//
// Copied in pieces, each followed by a launch that moves it, the first layer waits for the last piece's copy, its launch, its trip
// over the bus and a launch that packs; and every piece costs the bus the gap between two launches (2.4 MB in four pieces: 72 us where
// the bus needs 42; 0.8 MB in three: 45 us).  Here one launch is issued before the copy begins.  Its workgroups
// take bands of rows in the order of the copy, wait until the host has copied a band's rows of all channels, read them in 16-byte
// granules into LDS and write the packed rows.
// The host counts chunks of rows in a word of pinned memory.  Only the first workgroup reads that word (a trip over the bus); it
// repeats the count in device memory, where the others look.  Every wait is bounded: a launch that gives up writes nothing
// more, sets *error_host and ends.
// Bound by the bus, or by the host's copy where its source is not in the CPU's caches (44 GB/s).  64 workgroups with 6 KiB in flight each:
// the bus carries 52 to 55 GB/s for 256 KiB in flight and 42 to 46 for a megabyte (256 workgroups: ResNet-50 at batch 50 1 016 us a call,
// 64 982, 32 1 037).
#include <algorithm>

#include "conv_mfma.h"

namespace cvmhip {

constexpr int IMPORT_THREADS = 256, IMPORT_GROUPS = 64, IMPORT_BAND = 6144, IMPORT_CHUNK = 65536, IMPORT_LDS_MOST = 48 * 1024;
constexpr uint32_t IMPORT_GIVEN_UP = 0xffffffffu;

struct ImportStem {
  const int8_t* src;
  uint32_t* xs;
  int n, c, h, w, hp, wp, ph, pw, range;
  int band, bands, rows, chunks;   // packed rows of a band, bands and chunks of an image, image rows of a chunk
  int segment, granules;           // a channel's rows of a band in LDS: bytes, 16-byte granules at most
  int64_t slack_at, slack_end;     // words behind the last image, cleared
  FastDiv div_wp, div_bands;
  const uint64_t* progress_host;
  uint64_t* progress_dev;
  uint32_t* error_host;
  uint32_t ticket;
  uint64_t patience;               // of the first workgroup, in ticks of 10 ns; the others wait twice as long for it
};

// `need` chunks copied: thread 0 waits for all
__device__ __forceinline__ bool import_wait(const ImportStem& a, uint32_t need, int* s_go) {
  if (threadIdx.x == 0) {
    const uint64_t began = wall_clock64();
    int go = 0;
    for (;;) {
      const uint64_t v = __hip_atomic_load(a.progress_dev, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if ((uint32_t)(v >> 32) == a.ticket) {
        if ((uint32_t)v == IMPORT_GIVEN_UP) break;
        if ((uint32_t)v >= need) { go = 1; break; }
      }
      if (wall_clock64() - began > 2 * a.patience + 100000) {
        __hip_atomic_store(a.error_host, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        break;
      }
      __builtin_amdgcn_s_sleep(4);
    }
    *s_go = go;
  }
  __syncthreads();
  return *s_go != 0;
}

__global__ void __launch_bounds__(IMPORT_THREADS) k_import_stem(const ImportStem a) {
  extern __shared__ __attribute__((aligned(16))) int8_t s_rows[];   // [channel][segment]
  __shared__ int s_go;
  const int tid = threadIdx.x;
  if (blockIdx.x == 0) {
    if (tid != 0) return;
    const uint32_t total = (uint32_t)(a.n * a.chunks);
    const uint64_t began = wall_clock64();
    for (uint32_t seen = 0; seen < total;) {   // (no patience at all gives up whatever the host has copied)
      const uint64_t v = __hip_atomic_load(a.progress_host, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      if ((uint32_t)(v >> 32) == a.ticket && (uint32_t)v > seen && a.patience != 0) {
        seen = (uint32_t)v;
        __hip_atomic_store(a.progress_dev, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      } else if (wall_clock64() - began >= a.patience) {
        __hip_atomic_store(a.error_host, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(a.progress_dev, (uint64_t)a.ticket << 32 | IMPORT_GIVEN_UP, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
    }
    return;
  }
  const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(a.src), 0, 0x7fffffff, 0x00020000);
  typedef unsigned v4u __attribute__((ext_vector_type(4)));
  typedef unsigned v4w __attribute__((ext_vector_type(4), aligned(4)));
  for (int b = blockIdx.x - 1; b < a.n * a.bands; b += gridDim.x - 1) {
    const int img = (int)fastdiv((unsigned)b, a.div_bands), p0 = (b - img * a.bands) * a.band;
    const int p1 = p0 + a.band < a.hp ? p0 + a.band : a.hp;
    // image rows of the band
    const int y0 = p0 - a.ph < 0 ? 0 : p0 - a.ph, y1 = p1 - a.ph < a.h ? p1 - a.ph : a.h;
    int shift[4] = {0, 0, 0, 0};   // of a channel's first byte in its first granule
    if (y1 > y0) {
      if (!import_wait(a, (uint32_t)(img * a.chunks + (y1 - 1) / a.rows + 1), &s_go)) return;
      int64_t first[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int64_t at = ((int64_t)(img * a.c + (c < a.c ? c : 0)) * a.h + y0) * a.w;
        shift[c] = (int)(at & 15);
        first[c] = at - shift[c];
      }
      const int bytes = (y1 - y0) * a.w;
      for (int t0 = tid; t0 < a.c * a.granules; t0 += 4 * IMPORT_THREADS) {
        v4u v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int t = t0 + u * IMPORT_THREADS, c = (t >= a.granules) + (t >= 2 * a.granules) + (t >= 3 * a.granules), k = t - c * a.granules;
          const int64_t at = (c == 0 ? first[0] : c == 1 ? first[1] : c == 2 ? first[2] : first[3]) + 16 * k;
          const int sh = c == 0 ? shift[0] : c == 1 ? shift[1] : c == 2 ? shift[2] : shift[3];
          // (system scope: what another wait saw of this line, or an earlier launch, is not what is there now)
          if (c < a.c && 16 * k < sh + bytes) v[u] = __builtin_amdgcn_raw_buffer_load_b128(src, (int)at, 0, 17);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int t = t0 + u * IMPORT_THREADS, c = (t >= a.granules) + (t >= 2 * a.granules) + (t >= 3 * a.granules), k = t - c * a.granules;
          const int sh = c == 0 ? shift[0] : c == 1 ? shift[1] : c == 2 ? shift[2] : shift[3];
          if (c < a.c && 16 * k < sh + bytes) *reinterpret_cast<v4u*>(s_rows + c * a.segment + 16 * k) = v[u];
        }
      }
      __syncthreads();
    }
    uint32_t* out = a.xs + ((int64_t)img * a.hp + p0) * a.wp;
    const int words = (p1 - p0) * a.wp;
    for (int i = tid * 4; i < words; i += IMPORT_THREADS * 4) {
      int p = (int)fastdiv((unsigned)i, a.div_wp), q = i - p * a.wp;
      uint32_t d[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int y = p0 + p - a.ph, x = q - a.pw;
        const bool inside = y >= y0 && y < y1 && x >= 0 && x < a.w;
        const int at = inside ? (y - y0) * a.w + x : 0;
        int z[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          z[c] = c < a.c ? (int)s_rows[c * a.segment + shift[c] + at] : 0;
          z[c] = z[c] > a.range ? a.range : (z[c] < -a.range ? -a.range : z[c]);
        }
        const uint32_t pack = (uint32_t)(uint8_t)z[0] | (uint32_t)(uint8_t)z[1] << 8 | (uint32_t)(uint8_t)z[2] << 16 | (uint32_t)(uint8_t)z[3] << 24;
        d[u] = inside ? pack : 0u;
        if (++q == a.wp) {
          q = 0;
          ++p;
        }
      }
      if (i + 4 <= words) {
        *reinterpret_cast<v4w*>(out + i) = v4w{d[0], d[1], d[2], d[3]};
      } else {
#pragma unroll
        for (int u = 0; u < 3; ++u)
          if (i + u < words) out[i + u] = d[u];
      }
    }
    if (b == a.n * a.bands - 1)
      for (int64_t i = a.slack_at + tid; i < a.slack_end; i += IMPORT_THREADS) a.xs[i] = 0;
    __syncthreads();   // the rows in LDS have been read
  }
}

static int import_band(int c, int w) { return std::max(1, std::min(64, IMPORT_BAND / (c * w))); }
static int import_segment(int c, int w) { return (import_band(c, w) * w + 31) / 16 * 16; }

}  // namespace cvmhip

using namespace cvmhip;

extern "C" {

int cvmhip_import_stem_rows(int n, int c, int h, int w) {
  if (n < 1 || c < 1 || c > 4 || h < 1 || w < 1 || (int64_t)n * c * h * w > INT32_MAX - 64 || c * import_segment(c, w) > IMPORT_LDS_MOST) return 0;
  return std::max(1, std::min(h, IMPORT_CHUNK / (c * w)));
}

int cvmhip_import_stem_i8(const void* src_host, int32_t range, void* xs, int n, int c, int h, int w, int kh, int kw, int stride_h, int stride_w,
                          int pad_h, int pad_w, const uint64_t* progress_host, uint64_t* progress_dev, uint32_t* error_host, uint32_t ticket,
                          uint32_t patience_us, void* stream) {
  const int rows = cvmhip_import_stem_rows(n, c, h, w);
  if (!src_host || ((uintptr_t)src_host & 15) || !xs || ((uintptr_t)xs & 15) || range < 0 || range > 127 || rows == 0 || !stem_eligible(c, kh, kw, 1, 1) ||
      cvmhip_stem_input_bytes(n, h, w, kh, kw, stride_h, stride_w, pad_h, pad_w) == 0 || !progress_host || ((uintptr_t)progress_host & 7) ||
      !progress_dev || ((uintptr_t)progress_dev & 7) || !error_host)
    return arg_error("import_stem_i8");
  const StemGeom sg = stem_geom(n, h, w, kh, kw, stride_h, stride_w, pad_h, pad_w);
  ImportStem a = {};
  a.src = reinterpret_cast<const int8_t*>(src_host);
  a.xs = reinterpret_cast<uint32_t*>(xs);
  a.n = n; a.c = c; a.h = h; a.w = w; a.hp = sg.hp; a.wp = sg.wp; a.ph = pad_h; a.pw = pad_w; a.range = range;
  a.band = import_band(c, w);
  a.bands = (sg.hp + a.band - 1) / a.band;
  a.rows = rows;
  a.chunks = (h + rows - 1) / rows;
  a.segment = import_segment(c, w);
  a.granules = a.segment / 16;
  a.slack_at = (int64_t)n * sg.hp * sg.wp;
  a.slack_end = (int64_t)(sg.bytes / 4);
  a.div_wp = make_fastdiv((uint32_t)sg.wp);
  a.div_bands = make_fastdiv((uint32_t)a.bands);
  a.progress_host = progress_host;
  a.progress_dev = progress_dev;
  a.error_host = error_host;
  a.ticket = ticket;
  a.patience = (uint64_t)patience_us * 100;
  if ((int64_t)n * a.bands > INT32_MAX || a.slack_end > INT32_MAX || (int64_t)n * a.chunks >= IMPORT_GIVEN_UP) return arg_error("import_stem_i8 size");
  const int bands = n * a.bands;
  k_import_stem<<<1 + std::min(bands, IMPORT_GROUPS), IMPORT_THREADS, c * a.segment, as_stream(stream)>>>(a);
  return check_launch("import_stem_i8");
}

}  // extern "C"
