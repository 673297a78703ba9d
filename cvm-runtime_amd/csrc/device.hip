// Device memory, streams and events behind plain C entry points, so the host
// runtime (plain C++) never sees a HIP type.
#include "hip_common.h"

using namespace cvmhip;

#define HIP_TRY(expr, what)                                         \
  do {                                                              \
    hipError_t e_ = (expr);                                         \
    if (e_ != hipSuccess) {                                         \
      set_error("%s: %s", what, hipGetErrorString(e_));             \
      return CVMHIP_ERR_RUNTIME;                                    \
    }                                                               \
  } while (0)

#include <string.h>
#include <chrono>
#include <map>
#include <string>
#include <vector>

namespace cvmhip {

namespace {
struct TimedLaunch { std::string name, desc; double work, bytes; hipEvent_t e0, e1; };
bool g_timing = false;
std::vector<TimedLaunch> g_launches;
}  // namespace

bool kernel_timing_enabled() { return g_timing; }

void kernel_timing_mark(const char* name, double work, double bytes, const char* desc, hipStream_t s, bool start) {
  if (start) {
    TimedLaunch t;
    t.name = name;
    t.desc = desc ? desc : "";
    t.work = work;
    t.bytes = bytes;
    if (hipEventCreate(&t.e0) != hipSuccess || hipEventCreate(&t.e1) != hipSuccess) return;
    hipEventRecord(t.e0, s);
    g_launches.push_back(t);
  } else if (!g_launches.empty()) {
    hipEventRecord(g_launches.back().e1, s);
  }
}

__global__ void __launch_bounds__(256) k_fill32(int32_t* p, int32_t v, size_t n) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}

// Device -> pinned host memory, and a word that says so.  Every workgroup makes its stores visible to the host, by one fence, before it
// counts itself out; the last one to count stores the ticket.  The host polls that word instead of waiting for the
// stream (7.5 us from launch to seen, against 11.7 us for a launch and a stream synchronisation, and no copy calls).
struct ExportArgs {
  const int32_t* src[CVMHIP_EXPORT_MAX];
  int32_t* dst[CVMHIP_EXPORT_MAX];
  int64_t words[CVMHIP_EXPORT_MAX];
  uint64_t* pieces[CVMHIP_EXPORT_MAX];
  int count;
};

// An array in pieces of CVMHIP_EXPORT_PIECE words: one of equal words goes over the bus as that word.  (The rows of a detector behind the
// kept ones are all -1: 590 KB of SSD-512, 20.8 us from launch to seen, are there
// in 11.3, and the host fills what it would have copied: a call 243 -> 223 us.  590 KB of different words take 20.9.)
// A wavefront takes a piece, EXPORT_AHEAD of them where there are so many, all loaded before it asks about the first.
constexpr int EXPORT_AHEAD = 2;
__device__ __forceinline__ void export_pieces(const int32_t* src, int32_t* dst, uint64_t* pieces, int64_t words) {
  const int64_t whole = words / CVMHIP_EXPORT_PIECE, wavefronts = (int64_t)gridDim.x * 4;
  const int lane = threadIdx.x & 63;
  for (int64_t c0 = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); c0 < whole; c0 += wavefronts * EXPORT_AHEAD) {
    int4 v[EXPORT_AHEAD][4];
#pragma unroll
    for (int k = 0; k < EXPORT_AHEAD; ++k) {
      const int64_t c = c0 + k * wavefronts;
      if (c < whole)
#pragma unroll
        for (int q = 0; q < 4; ++q) v[k][q] = *reinterpret_cast<const int4*>(src + c * CVMHIP_EXPORT_PIECE + (q * 64 + lane) * 4);
    }
#pragma unroll
    for (int k = 0; k < EXPORT_AHEAD; ++k) {
      const int64_t c = c0 + k * wavefronts;
      if (c >= whole) break;   // (the same for all lanes)
      const int32_t first = __builtin_amdgcn_readfirstlane(v[k][0].x);
      bool same = true;
#pragma unroll
      for (int q = 0; q < 4; ++q) same = same && v[k][q].x == first && v[k][q].y == first && v[k][q].z == first && v[k][q].w == first;
      same = __all(same);
      if (!same)
#pragma unroll
        for (int q = 0; q < 4; ++q) *reinterpret_cast<int4*>(dst + c * CVMHIP_EXPORT_PIECE + (q * 64 + lane) * 4) = v[k][q];
      if (lane == 0) pieces[c] = ((uint64_t)same << 32) | (uint32_t)first;
    }
  }
  if (blockIdx.x == gridDim.x - 1)
    for (int64_t i = whole * CVMHIP_EXPORT_PIECE + threadIdx.x; i < words; i += 256) dst[i] = src[i];
}

template <bool PIECES>
__global__ void __launch_bounds__(256) k_export(ExportArgs a, const uint32_t* __restrict__ status, uint32_t* __restrict__ status_host,
                                                uint32_t* __restrict__ counter, uint32_t* __restrict__ flag) {
  const uint32_t ticket = threadIdx.x == 0 ? counter[1] + 1 : 0;   // (written by the last workgroup of the export before)
  const int64_t first = (int64_t)blockIdx.x * 256 + threadIdx.x, stride = (int64_t)gridDim.x * 256;
  for (int k = 0; k < a.count; ++k) {
    if (PIECES && a.pieces[k]) {
      export_pieces(a.src[k], a.dst[k], a.pieces[k], a.words[k]);
      continue;
    }
    const int64_t granules = a.words[k] / 4;
    const int4* s = reinterpret_cast<const int4*>(a.src[k]);
    int4* d = reinterpret_cast<int4*>(a.dst[k]);
    for (int64_t i = first; i < granules; i += stride) d[i] = s[i];
    const int64_t at = granules * 4 + first;
    if (at < a.words[k]) a.dst[k][at] = a.src[k][at];
  }
  if (status && blockIdx.x == 0 && threadIdx.x == 0) *status_host = *status;
  stores_done_barrier();
  if (threadIdx.x == 0) {
    __threadfence_system();
    const uint32_t before = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    if (before == gridDim.x - 1) {
      counter[0] = 0;
      counter[1] = ticket;
      __hip_atomic_store(flag, ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

}  // namespace cvmhip

extern "C" {

int cvmhip_device_count(int* count) {
  if (!count) return arg_error("device_count");
  HIP_TRY(hipGetDeviceCount(count), "hipGetDeviceCount");
  return CVMHIP_OK;
}

int cvmhip_set_device(int device_id) {
  HIP_TRY(hipSetDevice(device_id), "hipSetDevice");
  return CVMHIP_OK;
}

int cvmhip_alloc(void** ptr, size_t bytes) {
  if (!ptr) return arg_error("alloc");
  HIP_TRY(hipMalloc(ptr, bytes ? bytes : 256), "hipMalloc");
  return CVMHIP_OK;
}

int cvmhip_free(void* ptr) {
  if (ptr) HIP_TRY(hipFree(ptr), "hipFree");
  return CVMHIP_OK;
}

// A fill kernel rather than hipMemsetAsync so the call stays valid inside a captured graph.
int cvmhip_memset32(void* ptr, int32_t value, size_t count, void* stream) {
  if (count == 0) return CVMHIP_OK;
  if (!ptr) return arg_error("memset32");
  k_fill32<<<grid_for((int64_t)count, 256), 256, 0, as_stream(stream)>>>((int32_t*)ptr, value, count);
  return check_launch("memset32");
}

int cvmhip_host_alloc(void** ptr, size_t bytes) {
  if (!ptr) return arg_error("host_alloc");
  HIP_TRY(hipHostMalloc(ptr, bytes ? bytes : 256, hipHostMallocDefault), "hipHostMalloc");
  return CVMHIP_OK;
}

int cvmhip_host_free(void* ptr) {
  if (ptr) HIP_TRY(hipHostFree(ptr), "hipHostFree");
  return CVMHIP_OK;
}

// int8 -> int32 with the input clamp of the graph runtime (graph_runtime.cc:345-352)
__global__ void __launch_bounds__(256) k_widen_clamp(const int8_t* __restrict__ src, int32_t* __restrict__ dst, int64_t count,
                                                     int32_t range) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) {
    const int32_t v = src[i];
    dst[i] = v > range ? range : (v < -range ? -range : v);
  }
}

int cvmhip_widen_clamp_i8(const void* src, int32_t* dst, int64_t count, int32_t range, void* stream) {
  if (!src || !dst || count < 0 || range < 0) return arg_error("widen_clamp_i8");
  if (count == 0) return CVMHIP_OK;
  k_widen_clamp<<<grid_for(count, 256), 256, 0, as_stream(stream)>>>(reinterpret_cast<const int8_t*>(src), dst, count, range);
  return check_launch("widen_clamp_i8");
}

// plain 16-bytes-per-lane copy
__global__ void __launch_bounds__(256) k_copy16(const int4* __restrict__ src, int4* __restrict__ dst, int64_t count) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) dst[i] = src[i];
}

int cvmhip_copy_kernel(void* dst, const void* src, size_t bytes, void* stream) {
  if (!dst || !src || (bytes & 15) || ((uintptr_t)dst & 15) || ((uintptr_t)src & 15)) return arg_error("copy_kernel: 16-byte granules");
  if (bytes == 0 || dst == src) return CVMHIP_OK;
  const int64_t count = (int64_t)(bytes / 16);
  int64_t blocks = (count + 255) / 256;
  if (blocks > 256 * 32) blocks = 256 * 32;
  k_copy16<<<(unsigned)blocks, 256, 0, as_stream(stream)>>>(reinterpret_cast<const int4*>(src), reinterpret_cast<int4*>(dst), count);
  return check_launch("copy_kernel");
}

// Pinned host memory -> device.  Bound by the bus: four 16-byte requests per thread in flight move 46 GB/s (one request
// per thread: 42); the copy engine moves 59 GB/s, but the first kernel behind it waits about 10 us for its signal, and a
// piece costs the engine 5 us (2.4 MB in four pieces behind the host's copy of each: 65 us to the first kernel here, 90 us
// with the engine; 150 KB: 7 against 17 us).
__global__ void __launch_bounds__(256) k_import(const int4* __restrict__ src, int4* __restrict__ dst, int64_t count, int tail) {
  const int64_t i = (int64_t)blockIdx.x * 1024 + threadIdx.x;
  int4 v[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) v[u] = src[i + u * 256 < count ? i + u * 256 : count - 1];
#pragma unroll
  for (int u = 0; u < 4; ++u)
    if (i + u * 256 < count) dst[i + u * 256] = v[u];
  if (blockIdx.x == 0 && (int)threadIdx.x < tail)
    reinterpret_cast<int8_t*>(dst + count)[threadIdx.x] = reinterpret_cast<const int8_t*>(src + count)[threadIdx.x];
}

__global__ void __launch_bounds__(64) k_import_small(const int8_t* __restrict__ src, int8_t* __restrict__ dst, int count) {
  if ((int)threadIdx.x < count) dst[threadIdx.x] = src[threadIdx.x];
}

int cvmhip_import_bytes(void* dst, const void* src_host, size_t bytes, void* stream) {
  if (bytes == 0) return CVMHIP_OK;
  if (!dst || !src_host || ((uintptr_t)dst & 15) || ((uintptr_t)src_host & 15)) return arg_error("import_bytes");
  const int64_t count = (int64_t)(bytes / 16);
  const int tail = (int)(bytes % 16);
  if (count == 0)
    k_import_small<<<1, 64, 0, as_stream(stream)>>>(reinterpret_cast<const int8_t*>(src_host), reinterpret_cast<int8_t*>(dst), tail);
  else
    k_import<<<(unsigned)((count + 1023) / 1024), 256, 0, as_stream(stream)>>>(reinterpret_cast<const int4*>(src_host),
                                                                               reinterpret_cast<int4*>(dst), count, tail);
  return check_launch("import_bytes");
}

int cvmhip_export_words(const void* const* src, void* const* dst_host, const int64_t* words, int count, const uint32_t* status,
                        uint32_t* status_host, uint32_t* counter, uint32_t* flag_host, void* stream) {
  return cvmhip_export_pieces(src, dst_host, nullptr, words, count, status, status_host, counter, flag_host, stream);
}

int cvmhip_export_pieces(const void* const* src, void* const* dst_host, uint64_t* const* pieces_host, const int64_t* words, int count,
                         const uint32_t* status, uint32_t* status_host, uint32_t* counter, uint32_t* flag_host, void* stream) {
  if (!src || !dst_host || !words || count < 0 || count > CVMHIP_EXPORT_MAX || !counter || !flag_host || (status && !status_host))
    return arg_error("export_words");
  ExportArgs a{};
  int64_t most = 0;
  bool any = false;
  a.count = count;
  for (int k = 0; k < count; ++k) {
    if (!src[k] || !dst_host[k] || words[k] < 0 || ((uintptr_t)src[k] & 15) || ((uintptr_t)dst_host[k] & 15)) return arg_error("export_words");
    a.src[k] = reinterpret_cast<const int32_t*>(src[k]);
    a.dst[k] = reinterpret_cast<int32_t*>(dst_host[k]);
    a.words[k] = words[k];
    a.pieces[k] = pieces_host ? pieces_host[k] : nullptr;
    if ((uintptr_t)a.pieces[k] & 7) return arg_error("export_words");
    any = any || a.pieces[k];
    if (words[k] > most) most = words[k];
  }
  // 64 workgroups fill the bus
  int64_t blocks = (most / 4 + 255) / 256;
  if (blocks < 1) blocks = 1;
  if (blocks > 64) blocks = 64;
  if (any) k_export<true><<<(unsigned)blocks, 256, 0, as_stream(stream)>>>(a, status, status_host, counter, flag_host);
  else k_export<false><<<(unsigned)blocks, 256, 0, as_stream(stream)>>>(a, status, status_host, counter, flag_host);
  return check_launch("export_words");
}

int cvmhip_export_wait(const uint32_t* flag_host, uint32_t ticket, void* stream) {
  if (!flag_host) return arg_error("export_wait");
  // a run is milliseconds at most; past 50 ms the wait goes to the runtime, which also sees errors
  const auto began = std::chrono::steady_clock::now();
  for (uint32_t spin = 1;; ++spin) {
    if (__atomic_load_n(flag_host, __ATOMIC_ACQUIRE) == ticket) return CVMHIP_OK;
    if ((spin & 1023u) == 0 && std::chrono::steady_clock::now() - began > std::chrono::milliseconds(50)) break;
    __builtin_ia32_pause();
  }
  HIP_TRY(hipStreamSynchronize(as_stream(stream)), "export_wait");
  if (__atomic_load_n(flag_host, __ATOMIC_ACQUIRE) == ticket) return CVMHIP_OK;
  set_error("export_wait: the stream ended without the outputs");
  return CVMHIP_ERR_RUNTIME;
}

int cvmhip_copy_h2d(void* dst, const void* src, size_t bytes, void* stream) {
  if (bytes == 0) return CVMHIP_OK;
  HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, as_stream(stream)), "copy_h2d");
  return CVMHIP_OK;
}

int cvmhip_copy_d2h(void* dst, const void* src, size_t bytes, void* stream) {
  if (bytes == 0) return CVMHIP_OK;
  HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, as_stream(stream)), "copy_d2h");
  return CVMHIP_OK;
}

int cvmhip_copy_d2d(void* dst, const void* src, size_t bytes, void* stream) {
  if (bytes == 0 || dst == src) return CVMHIP_OK;
  HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, as_stream(stream)), "copy_d2d");
  return CVMHIP_OK;
}

int cvmhip_stream_create(void** stream) {
  if (!stream) return arg_error("stream_create");
  hipStream_t s;
  HIP_TRY(hipStreamCreate(&s), "hipStreamCreate");  // default priority
  *stream = s;
  return CVMHIP_OK;
}

int cvmhip_stream_destroy(void* stream) {
  if (stream) HIP_TRY(hipStreamDestroy(as_stream(stream)), "hipStreamDestroy");
  return CVMHIP_OK;
}

int cvmhip_stream_sync(void* stream) {
  HIP_TRY(hipStreamSynchronize(as_stream(stream)), "hipStreamSynchronize");
  return CVMHIP_OK;
}

// Timing is process-wide and meant for a single-threaded measurement harness.
int cvmhip_kernel_timing_begin(void) {
  g_launches.clear();
  g_timing = true;
  return CVMHIP_OK;
}

// Writes {"kernel": {"launches": n, "ms": total, "work": total}, ...}; with per_launch a list, in launch
// order, of {"kernel", "desc", "work", "bytes", "ms"}
static int timing_end(char* json_out, int capacity, bool per_launch) {
  g_timing = false;
  HIP_TRY(hipDeviceSynchronize(), "kernel_timing_end");
  struct Acc { long n = 0; double ms = 0, work = 0; };
  std::map<std::string, Acc> acc;
  std::string list = "[";
  for (TimedLaunch& t : g_launches) {
    float ms = 0;
    if (hipEventElapsedTime(&ms, t.e0, t.e1) == hipSuccess) {
      Acc& a = acc[t.name];
      a.n += 1;
      a.ms += ms;
      a.work += t.work;
      if (per_launch) {
        char buf[512];
        snprintf(buf, sizeof(buf), "%s{\"kernel\": \"%s\", \"desc\": \"%s\", \"work\": %.6e, \"bytes\": %.6e, \"ms\": %.6f}",
                 list.size() > 1 ? ", " : "", t.name.c_str(), t.desc.c_str(), t.work, t.bytes, ms);
        list += buf;
      }
    }
    hipEventDestroy(t.e0);
    hipEventDestroy(t.e1);
  }
  list += "]";
  g_launches.clear();
  std::string out = "{";
  bool first = true;
  for (const auto& kv : acc) {
    char buf[256];
    snprintf(buf, sizeof(buf), "%s\"%s\": {\"launches\": %ld, \"ms\": %.6f, \"work\": %.6e}", first ? "" : ", ",
             kv.first.c_str(), kv.second.n, kv.second.ms, kv.second.work);
    out += buf;
    first = false;
  }
  out += "}";
  const std::string& res = per_launch ? list : out;
  if (!json_out || (int)res.size() >= capacity) return arg_error("kernel_timing_end buffer");
  memcpy(json_out, res.c_str(), res.size() + 1);
  return CVMHIP_OK;
}

int cvmhip_kernel_timing_end(char* json_out, int capacity) { return timing_end(json_out, capacity, false); }

int cvmhip_kernel_timing_end_launches(char* json_out, int capacity) { return timing_end(json_out, capacity, true); }

int cvmhip_event_create(void** event) {
  if (!event) return arg_error("event_create");
  hipEvent_t e;
  HIP_TRY(hipEventCreate(&e), "hipEventCreate");
  *event = e;
  return CVMHIP_OK;
}

int cvmhip_event_destroy(void* event) {
  if (event) HIP_TRY(hipEventDestroy((hipEvent_t)event), "hipEventDestroy");
  return CVMHIP_OK;
}

int cvmhip_event_record(void* event, void* stream) {
  HIP_TRY(hipEventRecord((hipEvent_t)event, as_stream(stream)), "hipEventRecord");
  return CVMHIP_OK;
}

int cvmhip_device_sync(void) {
  HIP_TRY(hipDeviceSynchronize(), "hipDeviceSynchronize");
  return CVMHIP_OK;
}

int cvmhip_stream_wait_event(void* stream, void* event) {
  HIP_TRY(hipStreamWaitEvent(as_stream(stream), (hipEvent_t)event, 0), "hipStreamWaitEvent");
  return CVMHIP_OK;
}

int cvmhip_event_elapsed_ms(void* start, void* stop, float* ms) {
  HIP_TRY(hipEventSynchronize((hipEvent_t)stop), "hipEventSynchronize");
  HIP_TRY(hipEventElapsedTime(ms, (hipEvent_t)start, (hipEvent_t)stop), "hipEventElapsedTime");
  return CVMHIP_OK;
}

int cvmhip_kernel_timing_active(void) { return g_timing ? 1 : 0; }

int cvmhip_capture_begin(void* stream) {
  HIP_TRY(hipStreamBeginCapture(as_stream(stream), hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
  return CVMHIP_OK;
}

int cvmhip_capture_end(void* stream, void** graph_exec) {
  if (!graph_exec) return arg_error("capture_end");
  hipGraph_t graph = nullptr;
  HIP_TRY(hipStreamEndCapture(as_stream(stream), &graph), "hipStreamEndCapture");
  hipGraphExec_t exec = nullptr;
  hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  hipGraphDestroy(graph);
  if (e != hipSuccess) {
    set_error("hipGraphInstantiate: %s", hipGetErrorString(e));
    return CVMHIP_ERR_RUNTIME;
  }
  *graph_exec = exec;
  return CVMHIP_OK;
}

int cvmhip_graph_launch(void* graph_exec, void* stream) {
  HIP_TRY(hipGraphLaunch((hipGraphExec_t)graph_exec, as_stream(stream)), "hipGraphLaunch");
  return CVMHIP_OK;
}

int cvmhip_graph_destroy(void* graph_exec) {
  if (graph_exec) HIP_TRY(hipGraphExecDestroy((hipGraphExec_t)graph_exec), "hipGraphExecDestroy");
  return CVMHIP_OK;
}

}  // extern "C"
