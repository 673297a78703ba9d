// get_valid_counts and non_max_suppression for gfx950.
//
// Both are order-sensitive on the CPU; here the order is reproduced with
// wavefront ballots / prefix sums (stream compaction) and a rank sort whose key
// (score descending, original index ascending) is unique, so the result does
// not depend on scheduling.  Nothing is copied back to the host: valid_count is
// read on the device and every launch shape depends only on (batches, n, k).
#include <mutex>

#include "hip_common.h"

namespace cvmhip {

constexpr int GVC_CHUNK = 256;
// The kernels of this file are a handful of dependent round trips to memory and little else: whatever address does not depend on
// an earlier load is requested before that load is waited for, rows of up to ROW_REGS values among them.
constexpr int ROW_REGS = 8;
__device__ __forceinline__ void row_request(int32_t (&v)[ROW_REGS], const int32_t* __restrict__ row, int k) {
#pragma unroll
  for (int c = 0; c < ROW_REGS; ++c) v[c] = row[c < k ? c : k - 1];
}
__device__ __forceinline__ void row_store(int32_t* __restrict__ dst, const int32_t (&v)[ROW_REGS], const int32_t* __restrict__ row, int k) {
  if (k <= ROW_REGS) {
#pragma unroll
    for (int c = 0; c < ROW_REGS; ++c)
      if (c < k) dst[c] = v[c];
  } else {
    for (int c = 0; c < k; ++c) dst[c] = row[c];
  }
}

// number of rows in this 256-row chunk whose score passes the threshold
__global__ void __launch_bounds__(GVC_CHUNK)
k_gvc_count(const int32_t* __restrict__ x, int32_t* __restrict__ counts, int n, int k, int32_t thr, int nchunks) {
  __shared__ int wsum[GVC_CHUNK / 64];
  const int b = blockIdx.y, chunk = blockIdx.x;
  const int row = chunk * GVC_CHUNK + threadIdx.x;
  const bool keep = row < n && x[((int64_t)b * n + row) * k + 1] > thr;
  const unsigned long long m = __ballot(keep);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = __popcll(m);
  __syncthreads();
  if (threadIdx.x == 0) {
    int t = 0;
    for (int i = 0; i < GVC_CHUNK / 64; ++i) t += wsum[i];
    counts[b * nchunks + chunk] = t;
  }
}

// Each chunk derives its output offset from the counts of the chunks before it,
// then places its surviving rows in their original order; rows at or past the
// batch total are filled with -1.  OWN: there are no counts, every chunk counts all rows itself.
template <bool OWN>
__global__ void __launch_bounds__(GVC_CHUNK)
k_gvc_scatter(const int32_t* __restrict__ x, const int32_t* __restrict__ counts, int32_t* __restrict__ valid_count,
              int32_t* __restrict__ y, int n, int k, int32_t thr, int nchunks) {
  __shared__ int wsum[GVC_CHUNK / 64];
  __shared__ int s_bef[GVC_CHUNK / 64], s_tot[GVC_CHUNK / 64];
  __shared__ int s_before, s_total;
  const int b = blockIdx.y, chunk = blockIdx.x;
  const int row = chunk * GVC_CHUNK + threadIdx.x;
  const int32_t* src = x + ((int64_t)b * n + (row < n ? row : n - 1)) * k;
  const int32_t score = src[1];
  int32_t value[ROW_REGS];
  row_request(value, src, k);
  {
    // the counts are summed by all threads (one thread walking a hundred of them is a chain of a hundred loads)
    int before = 0, total = 0;
    if constexpr (OWN) {
      const int32_t* xb = x + (int64_t)b * n * k + 1;
      for (int c0 = 0; c0 < nchunks; c0 += 8) {
        int32_t v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int i = (c0 + u) * GVC_CHUNK + threadIdx.x;
          v[u] = xb[(int64_t)(i < n ? i : n - 1) * k];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int one = (c0 + u) * GVC_CHUNK + (int)threadIdx.x < n && v[u] > thr;
          before += c0 + u < chunk ? one : 0;
          total += one;
        }
      }
    } else {
      for (int c = threadIdx.x; c < nchunks; c += GVC_CHUNK) {
        const int v = counts[b * nchunks + c];
        before += c < chunk ? v : 0;
        total += v;
      }
    }
    before = wave_sum(before);
    total = wave_sum(total);
    if ((threadIdx.x & 63) == 0) { s_bef[threadIdx.x >> 6] = before; s_tot[threadIdx.x >> 6] = total; }
    __syncthreads();
    if (threadIdx.x == 0) {
      before = total = 0;
      for (int w = 0; w < GVC_CHUNK / 64; ++w) { before += s_bef[w]; total += s_tot[w]; }
      s_before = before;
      s_total = total;
      if (chunk == 0) valid_count[b] = total;
    }
  }
  const bool keep = row < n && score > thr;
  const unsigned long long m = __ballot(keep);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int in_wave = __popcll(m & ((1ull << lane) - 1ull));
  if (lane == 0) wsum[wv] = __popcll(m);
  __syncthreads();
  int pos = s_before + in_wave;
  for (int i = 0; i < wv; ++i) pos += wsum[i];
  int32_t* yb = y + (int64_t)b * n * k;
  if (keep) row_store(yb + (int64_t)pos * k, value, src, k);
  if (row < n && row >= s_total)
    for (int c = 0; c < k; ++c) yb[(int64_t)row * k + c] = -1;
}

// Up to so many chunks every chunk counts all rows itself, which saves the launch that counts: 1 000 rows 5.2 -> 3.2 us, 5 000 5.4 -> 4.0, 8 000
// 5.5 -> 4.4; at 24 564 (96 chunks) reading all scores costs a workgroup 4 us more than the counts and 7.9 us in all against 5.1.
constexpr int GVC_OWN_CHUNKS = 32;

// ------------------------------------------------------------------ NMS
// int64 IoU*100 of two corner-format boxes, same arithmetic as the reference
// (src/runtime/cpu/ops/nms.cc:4-40).
__device__ __forceinline__ int64_t iou100(const int32_t* r1, const int32_t* r2) {
  const int64_t a1 = (int64_t)wsub(r1[2], r1[0]) * wsub(r1[3], r1[1]);
  const int64_t a2 = (int64_t)wsub(r2[2], r2[0]) * wsub(r2[3], r2[1]);
  const int64_t sum_area = (int64_t)((uint64_t)a1 + (uint64_t)a2);
  if (sum_area <= 0) return 0;
  const int32_t xr = r1[2] < r2[2] ? r1[2] : r2[2], xl = r1[0] > r2[0] ? r1[0] : r2[0];
  const int32_t yb = r1[3] < r2[3] ? r1[3] : r2[3], yt = r1[1] > r2[1] ? r1[1] : r2[1];
  int32_t w = wsub(xr, xl), h = wsub(yb, yt);
  if (w < 0) w = 0;
  if (h < 0) h = 0;
  int64_t overlap = (int64_t)h * w;
  int64_t uni = sum_area - overlap;
  if (uni <= 0) return 0;
  if (INT64_MAX / 100 < overlap) uni /= 100; else overlap *= 100;
  return overlap / uni;
}

// iou100(r1, r2) >= thr without the 64-bit division when the products are small
// enough to compare exactly: floor(100*o/u) >= t  <=>  100*o >= t*u  for u > 0.
__device__ __forceinline__ bool iou_at_least(const int32_t* r1, const int32_t* r2, int thr) {
  const int64_t a1 = (int64_t)wsub(r1[2], r1[0]) * wsub(r1[3], r1[1]);
  const int64_t a2 = (int64_t)wsub(r2[2], r2[0]) * wsub(r2[3], r2[1]);
  const int64_t sum_area = (int64_t)((uint64_t)a1 + (uint64_t)a2);
  const int32_t xr = r1[2] < r2[2] ? r1[2] : r2[2], xl = r1[0] > r2[0] ? r1[0] : r2[0];
  const int32_t yb = r1[3] < r2[3] ? r1[3] : r2[3], yt = r1[1] > r2[1] ? r1[1] : r2[1];
  int32_t w = wsub(xr, xl), h = wsub(yb, yt);
  if (w < 0) w = 0;
  if (h < 0) h = 0;
  const int64_t overlap = (int64_t)h * w;
  const int64_t uni = sum_area - overlap;
  const int64_t small = (int64_t)1 << 40;
  if (sum_area > 0 && sum_area < small && overlap < small && uni > 0 && thr > 0 && thr < (1 << 20))
    return overlap * 100 >= (int64_t)thr * uni;
  return iou100(r1, r2) >= thr;
}

__device__ __forceinline__ int clamp_vc(int vc, int n) { return vc > n ? n : (vc < 0 ? 0 : vc); }

// The reference returns from the whole call at the first batch without valid
// rows (nms.cc:76-79): that batch is filled with -1 and later batches are left
// untouched.  0 = process normally, 1 = this is that batch, 2 = skipped.
__device__ __forceinline__ int batch_state(const int32_t* valid_count, int b, int n) {
  for (int i = 0; i < b; ++i)
    if (clamp_vc(valid_count[i], n) <= 0) return 2;
  return clamp_vc(valid_count[b], n) <= 0 ? 1 : 0;
}

constexpr int NMS_CLASSES = 64;   // the candidate rows of a batch are dealt to workgroups by id
// counts of a batch: candidate rows per class, workgroups of a class that have tested their pairs (k_nms_walk), candidate rows whose
// first value is negative.  Cleared by a kernel in front of the one that moves the rows, which fills them.
constexpr int NMS_ARRIVED = NMS_CLASSES, NMS_NEGATIVE = 2 * NMS_CLASSES, NMS_TALLY = 2 * NMS_CLASSES + 1;

// ---- sorted order of the first vc rows under (score descending, index ascending), which is what std::stable_sort
// gives (nms.cc:89-91), for up to BIN_MAX_ROWS rows: the rows are dealt to bins by the leading bits of their score
// and ranked inside their bin by comparing (score, index) words, so no order of arrival matters.
//   k_nms_place   a workgroup per chunk of BIN_CHUNK rows counts all rows per bin (every chunk for itself: reading the
//                 scores again costs less than a launch that shares the counts), turns the counts into the positions of
//                 its own rows and writes their words into their bins, in any order
//   k_nms_order   a thread per word counts the larger words of its bin, which makes its sorted slot, and moves its row
// Scores of magnitude below BIN_EXACT have bins of their own; beyond, a bin is a sign, the position of the leading one
// and three bits behind it (of the complement for negative scores): fixed, so no pass has to find the scores' range.
// The rows of a chunk lie together in a bin, so in a bin of one score (8-bit detectors saturate: hundreds of rows at 127)
// a word is only compared with the words of its own chunk; the rows of earlier chunks are in front by their counts.
// 9 000 rows with 8-bit scores: 9 us against 27 us for counting all pairs and moving the rows, and 75 us for the
// twelve launches of the radix sort below.  k_nms_place is bound by the lines of the rows that each workgroup pulls in for their scores
// (24 KiB a chunk at 64 bytes a clock: 5 900 of its 10 900 clocks), then by the chain of its sums; k_nms_order by round trips.  Rows that share one bin (all scores equal) cost n^2 comparisons spread
// over the chip, which stays below the sort's time up to BIN_MAX_ROWS.
constexpr int BIN_COUNT = 1024, BIN_CHUNK = 1024, BIN_MAX_ROWS = 32767, BIN_STAGE = 2048, BIN_EXACT = 256;

// 0 = the highest scores
__device__ __forceinline__ int score_bin(int32_t score) {
  const uint32_t v = (uint32_t)(score < 0 ? ~score : score);
  const int e = 31 - __clz((int)(v | 256u));
  const int at = v < BIN_EXACT ? (int)v : BIN_EXACT + (e - 8) * 8 + (int)((v >> (e - 3)) & 7u);   // at most 256 + 22 * 8 + 7 = 439
  return score < 0 ? 440 + at : 439 - at;
}

__device__ __forceinline__ unsigned long long score_word(int32_t score, int row) {
  return ((unsigned long long)((uint32_t)score ^ 0x80000000u) << 32) | (uint32_t)~(uint32_t)row;
}

// first[bin]: position of the bin's first word; mine[chunk][bin]: of its first word out of this chunk
__global__ void __launch_bounds__(BIN_CHUNK)
k_nms_place(const int32_t* __restrict__ x, const int32_t* __restrict__ valid_count, int32_t* __restrict__ mine,
            int32_t* __restrict__ first, unsigned long long* __restrict__ words, int32_t* __restrict__ tally, int n, int k, int score_index) {
  // rows of earlier chunks, of the others; four copies for the lanes, because 64 lanes on some sixty bins meet five at a time
  // (one copy: 4 000 clocks for 11 chunks), at an odd distance in banks
  constexpr int COPY = BIN_COUNT + 16;
  __shared__ int s_before[4 * COPY], s_rest[4 * COPY];
  __shared__ __attribute__((aligned(16))) int s_sum[BIN_CHUNK / 64];
  const int b = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int32_t* xb = x + (int64_t)b * n * k + score_index;
  const int chunk = blockIdx.x, row = chunk * BIN_CHUNK + tid;
  const int32_t score = xb[(int64_t)(row < n ? row : n - 1) * k];
  int32_t v[8];
  auto request = [&](int c0, int rows) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = (c0 + u) * BIN_CHUNK + tid;
      v[u] = xb[(int64_t)(i < rows ? i : rows - 1) * k];
    }
  };
  request(0, n);
  for (int t = tid; t < 4 * COPY; t += BIN_CHUNK) s_before[t] = s_rest[t] = 0;
  if (chunk == 0 && tid < NMS_TALLY) tally[b * NMS_TALLY + tid] = 0;
  if (batch_state(valid_count, b, n) != 0) return;
  const int vc = clamp_vc(valid_count[b], n);
  const int chunks = (vc + BIN_CHUNK - 1) / BIN_CHUNK;
  if (chunk >= chunks) return;
  __syncthreads();
  for (int c0 = 0; c0 < chunks; c0 += 8) {
    int bin[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) bin[u] = score_bin(v[u]) + (lane & 3) * COPY;
    if (c0 + 8 < chunks) request(c0 + 8, vc);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if ((c0 + u) * BIN_CHUNK + tid < vc) atomicAdd(c0 + u < chunk ? &s_before[bin[u]] : &s_rest[bin[u]], 1);
  }
  __syncthreads();
  int before = 0, total = 0;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    before += s_before[tid + c * COPY];
    total += s_rest[tid + c * COPY];
  }
  total += before;
  const int run = wave_scan_add(total);
  if (lane == 63) s_sum[wave] = run;
  __syncthreads();
  int sums[BIN_CHUNK / 64], start = run - total;
#pragma unroll
  for (int w = 0; w < BIN_CHUNK / 64; ++w) sums[w] = s_sum[w];
#pragma unroll
  for (int w = 0; w < BIN_CHUNK / 64; ++w) start += w < wave ? sums[w] : 0;
  s_before[tid] = start + before;
  __syncthreads();
  if (row < vc) words[(int64_t)b * n + atomicAdd(&s_before[score_bin(score)], 1)] = score_word(score, row);
  // (behind the barriers, which wait for a wavefront's stores as well)
  if (chunk == 0) first[(int64_t)b * (BIN_COUNT + 1) + tid] = start;
  if (chunk == 0 && tid == 0) first[(int64_t)b * (BIN_COUNT + 1) + BIN_COUNT] = vc;
  mine[((int64_t)b * gridDim.x + chunk) * BIN_COUNT + tid] = start + before;
}

// ---- ranks by a stable sort, for many rows.  Counting, for every row, the rows that sort
// before it costs n^2 comparisons (hours at the 2^24 rows the operator accepts); a least-significant-digit radix
// sort is the same stable order in four passes over the keys.  key = ~(score ^ 0x80000000) sorts ascending as the
// score sorts descending, and equal keys keep their order of arrival, i.e. ascending row index -- the order
// std::stable_sort gives (nms.cc:89-91).  A pass over one 8-bit digit is three launches:
//   k_radix_hist     every workgroup counts the digits of its RADIX_CHUNK consecutive elements
//   k_radix_scan     one workgroup per batch turns hist[digit][workgroup] into first positions (exclusive sum in
//                    digit-major order)
//   k_radix_scatter  every workgroup moves its elements, in their order, to first position + what came before
// Everything is integer counts: no float, no order-dependent atomics, so the result is the same on every run.
// Pass 0 reads the scores from the tensor (row i is element i); the last pass writes rank[row] = position.
constexpr int RADIX_CHUNK = 2048, RADIX_THREADS = 256, RADIX_ROUNDS = RADIX_CHUNK / RADIX_THREADS;
constexpr int RADIX_MIN_ROWS = BIN_MAX_ROWS + 1;

__device__ __forceinline__ uint32_t radix_key(int32_t score) { return ~((uint32_t)score ^ 0x80000000u); }

__global__ void __launch_bounds__(RADIX_THREADS)
k_radix_hist(const int32_t* __restrict__ x, const int32_t* __restrict__ valid_count, const uint32_t* __restrict__ keys_in,
             int32_t* __restrict__ hist, int n, int k, int score_index, int pass, int nblocks, int64_t key_stride) {
  __shared__ int s_hist[256];
  const int b = blockIdx.y, blk = blockIdx.x, tid = threadIdx.x;
  if (batch_state(valid_count, b, n) != 0) return;
  const int vc = clamp_vc(valid_count[b], n);
  s_hist[tid] = 0;
  __syncthreads();
  const int base = blk * RADIX_CHUNK;
  const int32_t* xb = x + (int64_t)b * n * k;
  const uint32_t* kin = keys_in + b * key_stride;
  for (int r = 0; r < RADIX_ROUNDS; ++r) {
    const int i = base + r * RADIX_THREADS + tid;
    if (i < vc) {
      const uint32_t key = pass == 0 ? radix_key(xb[(int64_t)i * k + score_index]) : kin[i];
      atomicAdd(&s_hist[(key >> (8 * pass)) & 255u], 1);
    }
  }
  __syncthreads();
  hist[((int64_t)b * 256 + tid) * nblocks + blk] = s_hist[tid];
}

// exclusive prefix sum over the 256 * nblocks counts of a batch, in place
__global__ void __launch_bounds__(1024)
k_radix_scan(const int32_t* __restrict__ valid_count, int32_t* __restrict__ hist, int32_t* __restrict__ tally, int n, int nblocks) {
  __shared__ int s_sum[1024];
  const int b = blockIdx.x, tid = threadIdx.x;
  if (tid < NMS_TALLY) tally[b * NMS_TALLY + tid] = 0;
  if (batch_state(valid_count, b, n) != 0) return;
  int32_t* h = hist + (int64_t)b * 256 * nblocks;
  const int total = 256 * nblocks;
  const int per = (total + 1023) / 1024;
  const int lo = tid * per < total ? tid * per : total, hi = lo + per < total ? lo + per : total;
  int sum = 0;
  for (int i = lo; i < hi; ++i) sum += h[i];
  s_sum[tid] = sum;
  __syncthreads();
  // inclusive scan of the 1024 partial sums
  for (int d = 1; d < 1024; d <<= 1) {
    const int v = tid >= d ? s_sum[tid - d] : 0;
    __syncthreads();
    s_sum[tid] += v;
    __syncthreads();
  }
  int run = s_sum[tid] - sum;
  for (int i = lo; i < hi; ++i) {
    const int c = h[i];
    h[i] = run;
    run += c;
  }
}

__global__ void __launch_bounds__(RADIX_THREADS)
k_radix_scatter(const int32_t* __restrict__ x, const int32_t* __restrict__ valid_count, const uint32_t* __restrict__ keys_in,
                const int32_t* __restrict__ idx_in, uint32_t* __restrict__ keys_out, int32_t* __restrict__ idx_out,
                const int32_t* __restrict__ hist, int32_t* __restrict__ rank, int n, int k, int score_index, int pass,
                int nblocks, int64_t key_stride, int last) {
  __shared__ int s_first[256];      // next free position of every digit for this workgroup
  __shared__ int s_cnt[4][256];     // elements of the current round per wavefront and digit
  const int b = blockIdx.y, blk = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (batch_state(valid_count, b, n) != 0) return;
  const int vc = clamp_vc(valid_count[b], n);
  const int base = blk * RADIX_CHUNK;
  if (base >= vc) return;
  s_first[tid] = hist[((int64_t)b * 256 + tid) * nblocks + blk];
  const int32_t* xb = x + (int64_t)b * n * k;
  const uint32_t* kin = keys_in + b * key_stride;
  const int32_t* iin = idx_in + b * key_stride;
  const unsigned long long lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  for (int r = 0; r < RADIX_ROUNDS; ++r) {
    for (int w = 0; w < 4; ++w) s_cnt[w][tid] = 0;
    __syncthreads();
    const int i = base + r * RADIX_THREADS + tid;
    const bool live = i < vc;
    uint32_t key = 0;
    int row = 0;
    if (live) {
      key = pass == 0 ? radix_key(xb[(int64_t)i * k + score_index]) : kin[i];
      row = pass == 0 ? i : iin[i];
    }
    const unsigned digit = (key >> (8 * pass)) & 255u;
    // lanes of this wavefront that are live and hold the same digit
    unsigned long long same = __ballot(live);
#pragma unroll
    for (int bit = 0; bit < 8; ++bit) {
      const unsigned long long set = __ballot((digit >> bit) & 1u);
      same &= ((digit >> bit) & 1u) ? set : ~set;
    }
    const int before = __popcll(same & lt);
    if (live && before == 0) s_cnt[wave][digit] = __popcll(same);   // the first lane of every group of equal digits
    __syncthreads();
    if (live) {
      int pos = s_first[digit] + before;
      for (int w = 0; w < wave; ++w) pos += s_cnt[w][digit];
      if (last) {
        rank[(int64_t)b * n + row] = pos;
      } else {
        keys_out[b * key_stride + pos] = key;
        idx_out[b * key_stride + pos] = row;
      }
    }
    __syncthreads();
    s_first[tid] += s_cnt[0][tid] + s_cnt[1][tid] + s_cnt[2][tid] + s_cnt[3][tid];
    __syncthreads();
  }
}

// Row i moves to its sorted slot r; rows ranked at or past top_k are overwritten with -1 in the input tensor instead
// (nms.cc:92-96).  code[slot] = class of the row's id (bits 0..5) and whether its first value is negative (bit 8).
// Every candidate is counted in s_tally.
__device__ __forceinline__ void nms_move_row(int32_t* __restrict__ x, int32_t* __restrict__ code, int32_t* __restrict__ sorted, int* s_tally,
                                             const int32_t (&value)[ROW_REGS], int32_t id, int b, int n, int k, int i, int r, int topk) {
  int32_t* xrow = x + ((int64_t)b * n + i) * k;
  if (topk > 0 && r >= topk) {  // never looked at again
    for (int c = 0; c < k; ++c) xrow[c] = -1;
    return;
  }
  const int cls = id & (NMS_CLASSES - 1);
  code[(int64_t)b * n + r] = cls | (value[0] < 0 ? 256 : 0);
  row_store(sorted + ((int64_t)b * n + r) * k, value, xrow, k);
  atomicAdd(&s_tally[cls], 1);
  if (value[0] < 0) atomicAdd(&s_tally[NMS_CLASSES], 1);
}
__device__ __forceinline__ void nms_add_tally(const int* s_tally, int32_t* __restrict__ tally, int b) {
  __syncthreads();
  const int t = threadIdx.x;
  if (t <= NMS_CLASSES && s_tally[t]) atomicAdd(&tally[b * NMS_TALLY + (t < NMS_CLASSES ? t : NMS_NEGATIVE)], s_tally[t]);
}

// Every output row starts as -1: k_nms_emit writes the kept rows over the front.
__device__ __forceinline__ void nms_clear_rows(int32_t* __restrict__ y, int b, int n, int k, int row0) {
  const int rows = n - row0 < 256 ? n - row0 : 256;
  int32_t* at = y + ((int64_t)b * n + row0) * k;
  for (int t = threadIdx.x; t < rows * k; t += 256) at[t] = -1;
}

// ranks from the radix sort
__global__ void __launch_bounds__(256)
k_nms_scatter(int32_t* __restrict__ x, const int32_t* __restrict__ valid_count, const int32_t* __restrict__ rank,
              int32_t* __restrict__ code, int32_t* __restrict__ sorted, int32_t* __restrict__ y, int32_t* __restrict__ tally,
              int n, int k, int topk, int id_index) {
  const int b = blockIdx.y;
  const int state = batch_state(valid_count, b, n);
  if (state == 2) return;
  nms_clear_rows(y, b, n, k, blockIdx.x * 256);
  __shared__ int s_tally[NMS_CLASSES + 1];
  const int i = blockIdx.x * 256 + threadIdx.x, vc = clamp_vc(valid_count[b], n);
  if (state == 1 || (int)blockIdx.x * 256 >= vc) return;
  if (threadIdx.x <= NMS_CLASSES) s_tally[threadIdx.x] = 0;
  __syncthreads();
  if (i < vc) {
    int32_t value[ROW_REGS];
    const int32_t* xrow = x + ((int64_t)b * n + i) * k;
    row_request(value, xrow, k);
    const int32_t id = id_index >= 0 ? xrow[id_index] : 0;
    nms_move_row(x, code, sorted, s_tally, value, id, b, n, k, i, rank[(int64_t)b * n + i], topk);
  }
  nms_add_tally(s_tally, tally, b);
}

// words of p[from, to) that are larger than `me`, eight reads in flight
__device__ __forceinline__ int nms_count_above(const unsigned long long* p, int from, int to, unsigned long long me) {
  int c = 0, q = from;
  for (; q + 8 <= to; q += 8) {
    unsigned long long o[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) o[u] = p[q + u];
#pragma unroll
    for (int u = 0; u < 8; ++u) c += o[u] > me;
  }
  for (; q < to; ++q) c += p[q] > me;
  return c;
}

// ranks from the bins: the words of the bins that this workgroup's 256 words lie in pass through LDS when they fit
__global__ void __launch_bounds__(256)
k_nms_order(int32_t* __restrict__ x, const int32_t* __restrict__ valid_count, const int32_t* __restrict__ mine,
            const int32_t* __restrict__ first, const unsigned long long* __restrict__ words, int32_t* __restrict__ code,
            int32_t* __restrict__ sorted, int32_t* __restrict__ y, int32_t* __restrict__ tally, int n, int k, int topk, int id_index) {
  __shared__ unsigned long long s_word[BIN_STAGE];
  __shared__ int s_span[2], s_tally[NMS_CLASSES + 1];
  const int b = blockIdx.y, p0 = blockIdx.x * 256, tid = threadIdx.x;
  const unsigned long long* wb = words + (int64_t)b * n;
  const int32_t* fb = first + (int64_t)b * (BIN_COUNT + 1);
  unsigned long long me = wb[p0 + tid < n ? p0 + tid : n - 1];   // past the valid rows: whatever lies there, not used
  const int state = batch_state(valid_count, b, n);
  if (state == 2) return;
  const int vc = clamp_vc(valid_count[b], n);
  if (state == 1 || p0 >= vc) {
    nms_clear_rows(y, b, n, k, p0);
    return;
  }
  const bool live = p0 + tid < vc;
  if (!live) me = score_word(INT32_MIN, 0);
  const int32_t score = (int32_t)((uint32_t)(me >> 32) ^ 0x80000000u);
  const int bin = score_bin(score), row = live ? (int)~(uint32_t)me : 0;
  int lo = fb[bin], hi = fb[bin + 1];
  int32_t value[ROW_REGS];
  const int32_t* xrow = x + ((int64_t)b * n + row) * k;
  row_request(value, xrow, k);
  const int32_t id = id_index >= 0 ? xrow[id_index] : 0;
  const bool near = score < BIN_EXACT && ~score < BIN_EXACT;
  const int chunk = row / BIN_CHUNK;
  const int32_t* m = mine + ((int64_t)b * ((n + BIN_CHUNK - 1) / BIN_CHUNK) + chunk) * BIN_COUNT + bin;
  const bool more = (chunk + 1) * BIN_CHUNK < vc;
  const int own_lo = m[0], own_hi = m[more ? BIN_COUNT : 0];
  if (tid <= NMS_CLASSES) s_tally[tid] = 0;
  if (tid == 0) s_span[0] = lo;
  if (tid == (p0 + 255 < vc ? 255 : vc - 1 - p0)) s_span[1] = hi;
  __syncthreads();
  const int from = s_span[0], to = s_span[1];   // the bins of the workgroup's words
  const bool past = topk > 0 && lo >= topk;   // every row of this bin is past top_k: which rank it has is of no interest
  if (!past && hi - lo > 128 && near) {
    lo = own_lo;
    if (more) hi = own_hi;
  }
  int r = lo;
  if (to - from <= BIN_STAGE) {
    for (int t = from + tid; t < to; t += 256) s_word[t - from] = wb[t];
    __syncthreads();
    if (!past) r += nms_count_above(s_word, lo - from, hi - from, me);
  } else {
    if (!past) r += nms_count_above(wb, lo, hi, me);
  }
  if (live) nms_move_row(x, code, sorted, s_tally, value, id, b, n, k, row, r, topk);
  nms_add_tally(s_tally, tally, b);
  nms_clear_rows(y, b, n, k, p0);   // (behind the barriers, which wait for a wavefront's stores as well)
}

// ---- the greedy walk.  In sorted order a surviving row removes every later row with the same id that overlaps it
// enough, up to (not including) the first later row whose first value is negative (nms.cc:98-124).  Two facts take
// the walk apart:
//   * rows of different ids never meet, so the rows are dealt to NMS_CLASSES workgroups by the low bits of their id
//     (one workgroup when force_suppress or id_index < 0 makes every row meet every other);
//   * row i may remove row j > i only if no row in (i, j] starts with a negative value, i.e. if as many such rows
//     lie at or before i as at or before j.  That count (`seg`) is one more value two rows have to share.
// A workgroup lists its rows in sorted order and takes them 64 at a time: all wavefronts test the 64 rows against
// the rows kept so far (each wavefront a sixteenth of those; a lane is a row, the kept row is a broadcast from LDS)
// and, at the same time, the 64 against each other (one ballot per row); then one wavefront settles the block in a
// few rounds of ballots and appends the survivors.  Only kept rows are ever tested
// against, so the work is kept x rows / 2 per class instead of one dependent step per row.
// Bound by those tests when one class holds everything, otherwise by the two barriers of a block.  24 564 rows,
// 9 000 of them valid, 21 ids: 22.5 ms in the row-by-row walk of one workgroup, 29 us here, 15 us by the masks below; the first 400
// rows: 5 us.
constexpr int NMS_THREADS = 1024, NMS_WAVES = NMS_THREADS / 64;
constexpr int NMS_WINDOW = 1024;   // rows staged in LDS at a time
constexpr int NMS_KEPT = 2048;     // kept rows held in LDS; later ones are read from memory
constexpr uint32_t NMS_WIDE = 0xffffffffu;

struct __attribute__((aligned(16))) NmsRow {
  int32_t x1, y1, x2, y2;
  uint32_t part;     // threshold x area; NMS_WIDE: this box needs the test with 64-bit products
  int32_t id, seg;
  int32_t pos;       // sorted position; bit 31: the row starts with a negative value
};

__device__ __forceinline__ void nms_load_row(NmsRow& q, const int32_t* row, int coord_start, int id_index, int thr) {
  typedef int v4i __attribute__((ext_vector_type(4), aligned(4)));
  const v4i box = *reinterpret_cast<const v4i*>(row + coord_start);   // one request: the rows lie anywhere
  q.x1 = box[0];
  q.y1 = box[1];
  q.x2 = box[2];
  q.y2 = box[3];
  q.id = id_index >= 0 ? row[id_index] : 0;
  const int32_t lim = 1 << 20;
  const bool in = q.x1 >= -lim && q.x1 <= lim && q.y1 >= -lim && q.y1 <= lim && q.x2 >= -lim && q.x2 <= lim && q.y2 >= -lim && q.y2 <= lim;
  const int64_t w = (int64_t)q.x2 - q.x1, h = (int64_t)q.y2 - q.y1;
  // an empty box overlaps nothing: any part above zero keeps 0 >= part + part false
  q.part = !in || thr > 100 ? NMS_WIDE : (w <= 0 || h <= 0) ? 1u : w * h < (1 << 24) ? (uint32_t)(w * h) * (uint32_t)thr : NMS_WIDE;
}

// Same id and iou100(a, b) >= thr for two boxes that are not NMS_WIDE: floor(100 o / (A + B - o)) >= t is
// (100 + t) o >= t A + t B, and with areas below 2^24 and t <= 100 both sides stay below 2^32.  No branch and no
// product wider than 24 bits (those run at full rate).
__device__ __forceinline__ bool nms_hits(const NmsRow& a, const NmsRow& b, uint32_t scale) {
  const int32_t w = (a.x2 < b.x2 ? a.x2 : b.x2) - (a.x1 > b.x1 ? a.x1 : b.x1);
  const int32_t h = (a.y2 < b.y2 ? a.y2 : b.y2) - (a.y1 > b.y1 ? a.y1 : b.y1);
  const uint32_t o = __umul24(w > 0 ? w : 0, h > 0 ? h : 0);
  return (__umul24(o, scale) >= a.part + b.part) & (a.id == b.id);
}

// the same for any two rows
__device__ __forceinline__ bool nms_hits_any(const NmsRow& a, const NmsRow& b, int thr) {
  const int32_t ra[4] = {a.x1, a.y1, a.x2, a.y2}, rb[4] = {b.x1, b.y1, b.x2, b.y2};
  return a.id == b.id && a.seg == b.seg && iou_at_least(ra, rb, thr);
}

// The rows of a block that stay: `front` is the rows in front of this lane's row that would remove it (overlap is symmetric),
// `open` those that no earlier block has removed.  A row stays when none of the rows in front is kept or still open, and goes
// when one of them is kept: a few rounds settle the block (the first open row is settled in every round), where a walk
// takes a step per overlapping row.
__device__ __forceinline__ unsigned long long nms_settle(unsigned long long front, unsigned long long open, int lane) {
  unsigned long long stay = 0;
  while (open) {
    const bool mine = (open >> lane) & 1ull;
    const unsigned long long now = __ballot(mine && !(front & (stay | open)));
    stay |= now;
    open &= ~(now | __ballot(mine && (front & stay)));
  }
  return stay;
}

// ---- the walk of a class by overlap masks, for NMS_PAIRS_LEAST to NMS_PAIRS_MOST rows whose coordinates fit in 15 bits.
// Tested block by block a class costs 64 x (rows kept so far) tests and two barriers per block of 64 rows, all in one compute
// unit: 5 700 clocks a block, most of them the vector instructions of the tests.  Here all pairs of the class are tested first, by
// `parts` workgroups that each list the class for themselves, in packed 16-bit arithmetic, into a 64-bit mask per row and block of
// rows in front of it; the last of them to finish settles the blocks in order from the masks (a row is removed by a kept row of
// an earlier block: one AND per block), 900 clocks each.  11 000 rows of 21 ids: 28 -> 15 us (35 K clocks: 11 K list the class, 5 K load
// its rows, 4 K test, 8 K hand the masks over, 6 K settle); 1 000 rows that all meet: 66 -> 37 us.
constexpr int NMS_PAIRS_LEAST = 129, NMS_PAIRS_MOST = NMS_WINDOW;
constexpr int NMS_PAIRS_BLOCKS = NMS_PAIRS_MOST / 64, NMS_PAIRS_LDS = NMS_PAIRS_BLOCKS * (NMS_PAIRS_BLOCKS + 1) / 2 * 64 * 8;
constexpr int NMS_PAIRS_WORDS = 10;   // mask words per row of the class: b blocks have b (b + 1) / 2 * 64, at most 10 for every row of (b - 1) * 64 + 1

// box of a staged row in 16-bit halves: its NmsRow's x1 and y1 hold (x1, y1) and (x2, y2) while pairs are tested
typedef short nms_v2s __attribute__((ext_vector_type(2)));
__device__ __forceinline__ int32_t nms_pack(int32_t a, int32_t b) { return (int32_t)((uint32_t)(a & 0xffff) | ((uint32_t)b << 16)); }
__device__ __forceinline__ bool nms_fits16(const NmsRow& q) {
  auto in = [](int32_t v) { return v >= -16384 && v <= 16383; };   // differences fit in 16 bits
  return in(q.x1) && in(q.y1) && in(q.x2) && in(q.y2);
}

// A wavefront's share of the pairs of blocks (i, j), i <= j, half a pair at a time: bits of 32 rows of block i for every row of block j;
// inside a block only rows in front of a row count.  masks[pair][half][row of j].
__device__ __forceinline__ void nms_pairs(const NmsRow* rows, int total, int iou_threshold, uint32_t* __restrict__ masks, int unit, int units, int lane) {
  const int blocks = (total + 63) >> 6, all = blocks * (blocks + 1);
  const uint32_t scale = 100u + (uint32_t)iou_threshold;
  for (; unit < all; unit += units) {
    const int pair = unit >> 1;
    int j = 0;
    while ((j + 1) * (j + 2) / 2 <= pair) ++j;
    const int i = pair - j * (j + 1) / 2;
    const int mine = j * 64 + lane, from = i * 64 + (unit & 1) * 32;
    const NmsRow me = rows[mine < total ? mine : total - 1];
    const nms_v2s lo = __builtin_bit_cast(nms_v2s, me.x1), hi = __builtin_bit_cast(nms_v2s, me.y1), zero = {0, 0};
    uint32_t bits = 0;
#pragma unroll 8
    for (int t = 0; t < 32; ++t) {
      // (a row past the end repeats the last one: its bit stands behind every row of the block)
      const NmsRow& o = rows[from + t < total ? from + t : total - 1];
      const nms_v2s d = __builtin_elementwise_max(__builtin_elementwise_min(__builtin_bit_cast(nms_v2s, o.y1), hi) -
                                                  __builtin_elementwise_max(__builtin_bit_cast(nms_v2s, o.x1), lo), zero);
      const uint32_t side = __builtin_bit_cast(uint32_t, d), overlap = __umul24(side & 0xffffu, side >> 16);
      const bool hit = (__umul24(overlap, scale) >= o.part + me.part) & (o.id == me.id);
      bits |= (hit ? 1u : 0u) << t;
    }
    if (i == j) {
      const int ahead = lane - (unit & 1) * 32;
      bits &= ahead <= 0 ? 0u : ahead >= 32 ? ~0u : (1u << ahead) - 1u;
    }
    __hip_atomic_store(masks + unit * 64 + lane, bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

__global__ void __launch_bounds__(NMS_THREADS)
k_nms_walk(const int32_t* __restrict__ valid_count, const int32_t* __restrict__ sorted, const int32_t* __restrict__ code,
           int32_t* __restrict__ list, int32_t* __restrict__ kept, uint8_t* __restrict__ flags, int32_t* __restrict__ tally,
           uint32_t* __restrict__ masks, int64_t mask_words, int n, int k, int iou_threshold, int topk, int coord_start, int id_index,
           int by_class, int parts) {
  __shared__ NmsRow s_row[NMS_WINDOW];
  __shared__ NmsRow s_kept[NMS_PAIRS_LDS > NMS_KEPT * (int)sizeof(NmsRow) ? NMS_PAIRS_LDS / sizeof(NmsRow) : NMS_KEPT];   // or the masks
  __shared__ unsigned long long s_mask[64], s_dead[2];
  __shared__ int s_count[NMS_WAVES], s_neg[NMS_WAVES], s_k;
  const int b = blockIdx.y, cls = blockIdx.x / parts, part = blockIdx.x - cls * parts, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int32_t* tl = tally + b * NMS_TALLY;
  const int rows_of = tl[lane], cuts = __builtin_amdgcn_readfirstlane(tl[NMS_NEGATIVE]);
  if (batch_state(valid_count, b, n) != 0) return;
  const int vc = clamp_vc(valid_count[b], n);
  const int keep = (topk >= 0 && topk < vc) ? topk : vc;
  // candidates of this class, and of the classes in front of it
  const int total = by_class ? __builtin_amdgcn_readlane(rows_of, cls) : keep;
  if (total == 0) return;
  const int base = by_class ? __builtin_amdgcn_readlane(wave_scan_add(rows_of), cls) - total : 0;
  bool pairs = masks && total >= NMS_PAIRS_LEAST && total <= NMS_PAIRS_MOST && cuts == 0;
  if (!pairs && part != 0) return;
  const int32_t* srt = sorted + (int64_t)b * n * k;
  const int32_t* cd = code + (int64_t)b * n;
  uint8_t* fl = flags + (int64_t)b * n * 4;
  const unsigned long long lt = (1ull << lane) - 1ull;

  // this workgroup's rows in sorted order: every wavefront counts its own stretch of the codes, then lists it.  The first
  // NMS_CODES * 64 codes of a stretch stay in registers between the two.
  constexpr int NMS_CODES = 12;
  const int per = ((keep + NMS_WAVES - 1) / NMS_WAVES + 63) & ~63;
  const int lo = wave * per, hi = lo + per < keep ? lo + per : keep;
  int mine = 0, neg = 0;
  // the code of a row of this class has 0 in its low byte here, one past the end is 255
  auto request = [&](int p) { return cd[p + lane < hi ? p + lane : keep - 1]; };
  auto tell = [&](int c, int p) { return p + lane < hi ? (by_class ? c ^ cls : c & 256) : 255; };
  auto count = [&](int c) {
    mine += __popcll(__ballot((c & 255) == 0));
    if (cuts) neg += __popcll(__ballot(c >= 256));
  };
  int32_t held[NMS_CODES];
#pragma unroll
  for (int u = 0; u < NMS_CODES; ++u)
    if (lo + u * 64 < hi) held[u] = request(lo + u * 64);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < NMS_CODES; ++u)
    if (lo + u * 64 < hi) {
      held[u] = tell(held[u], lo + u * 64);
      count(held[u]);
    }
  for (int p0 = lo + NMS_CODES * 64; p0 < hi; p0 += 256) {
    int32_t c[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) c[u] = request(p0 + u * 64);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 4; ++u) count(tell(c[u], p0 + u * 64));
  }
  if (lane == 0) {
    s_count[wave] = mine;
    s_neg[wave] = neg;
  }
  if (tid < 2) s_dead[tid] = 0;
  __syncthreads();
  int at = 0, seg = 0;
#pragma unroll
  for (int w = 0; w < NMS_WAVES; ++w) {
    at += w < wave ? s_count[w] : 0;
    seg += w < wave ? s_neg[w] : 0;
  }
  // rows past the first window, and later the kept rows past NMS_KEPT, live in memory at this class's own stretch
  int32_t* ls = list + (int64_t)b * n + base;
  // (list: position of row t, kept: its seg; once row t is staged, kept row q <= t goes to the same slots)
  int32_t* kp = kept + (int64_t)b * n + base;
  auto enter = [&](int c, int p0) {
    const int p = p0 + lane;
    const bool own = (c & 255) == 0;
    const unsigned long long om = __ballot(own);
    const int t = at + __builtin_amdgcn_mbcnt_hi((uint32_t)(om >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)om, 0));
    at += __popcll(om);
    if (total <= NMS_WINDOW && !cuts) {
      if (own) s_row[t].pos = p;
      return;
    }
    const bool ng = c >= 256;
    const unsigned long long nm = __ballot(ng);
    if (own) {
      const int sg = seg + __popcll(nm & lt) + (ng ? 1 : 0);
      const int word = p | (ng ? (int)0x80000000u : 0);
      if (t < NMS_WINDOW) {
        s_row[t].pos = word;
        s_row[t].seg = sg;
      } else {
        ls[t] = word;
        kp[t] = sg;
      }
    }
    seg += __popcll(nm);
  };
#pragma unroll
  for (int u = 0; u < NMS_CODES; ++u)
    if (lo + u * 64 < hi) enter(held[u], lo + u * 64);
  for (int p0 = lo + NMS_CODES * 64; p0 < hi; p0 += 256) {
    int32_t c[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) c[u] = request(p0 + u * 64);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 4; ++u) enter(tell(c[u], p0 + u * 64), p0 + u * 64);
  }
  __syncthreads();

  if (pairs) {   // every part comes to the same decision
    NmsRow q;
    int unfit = 0;
    if (tid < total) {
      q.pos = s_row[tid].pos;
      q.seg = 0;
      nms_load_row(q, srt + (int64_t)q.pos * k, coord_start, id_index, iou_threshold);
      if (!by_class) q.id = 0;
      unfit = q.part == NMS_WIDE || !nms_fits16(q);
    }
    pairs = !__syncthreads_or(unfit);
    if (pairs) {
      if (tid < total) {
        const int32_t x1 = nms_pack(q.x1, q.y1), y1 = nms_pack(q.x2, q.y2);
        q.x1 = x1;
        q.y1 = y1;
        s_row[tid] = q;
      }
      uint32_t* own = masks + b * mask_words * 2 + (int64_t)base * (NMS_PAIRS_WORDS * 2);
      __syncthreads();
      nms_pairs(s_row, total, iou_threshold, own, part * NMS_WAVES + wave, parts * NMS_WAVES, lane);
      stores_done_barrier();
      if (parts > 1) {
        if (tid == 0) s_k = __hip_atomic_fetch_add(&tl[NMS_ARRIVED + cls], 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (s_k != parts - 1) return;
      }
      const int blocks = (total + 63) >> 6, halves = blocks * (blocks + 1) * 64;
      uint32_t* m = reinterpret_cast<uint32_t*>(s_kept);
      for (int t = tid; t < halves; t += NMS_THREADS) m[t] = __hip_atomic_load(own + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      if (wave != 0) return;
      auto mask = [&](int pair) { return (unsigned long long)m[pair * 128 + 64 + lane] << 32 | m[pair * 128 + lane]; };
      uint32_t kept_lo = 0, kept_hi = 0;   // lane i: the rows of block i that stay
      for (int j = 0; j < blocks; ++j) {
        const int first = j * (j + 1) / 2;
        uint32_t met = 0;
#pragma unroll 4
        for (int i = 0; i < j; ++i)
          met |= (m[(first + i) * 128 + lane] & (uint32_t)__builtin_amdgcn_readlane((int)kept_lo, i)) |
                 (m[(first + i) * 128 + 64 + lane] & (uint32_t)__builtin_amdgcn_readlane((int)kept_hi, i));
        const unsigned long long front = (unsigned long long)m[(first + j) * 128 + 64 + lane] << 32 | m[(first + j) * 128 + lane];
        const int t = j * 64 + lane;
        const unsigned long long stay = nms_settle(front, __ballot(t < total && met == 0), lane);
        if (lane == j) {
          kept_lo = (uint32_t)stay;
          kept_hi = (uint32_t)(stay >> 32);
        }
        if (t < total) fl[s_row[t].pos] = (stay >> lane) & 1ull;
      }
      return;
    }
    if (part != 0) return;
    __syncthreads();
  }

  int K = 0, turn = 0, wide = cuts != 0;
  const uint32_t scale = 100u + (uint32_t)iou_threshold;
  for (int w0 = 0; w0 < total; w0 += NMS_WINDOW) {
    const int rows = total - w0 < NMS_WINDOW ? total - w0 : NMS_WINDOW;
    int odd = 0;
    if (tid < rows) {
      NmsRow q;
      q.pos = w0 ? ls[w0 + tid] : s_row[tid].pos;
      q.seg = w0 ? kp[w0 + tid] : cuts ? s_row[tid].seg : 0;
      nms_load_row(q, srt + (int64_t)(q.pos & 0x7fffffff) * k, coord_start, id_index, iou_threshold);
      if (!by_class) q.id = 0;
      odd = q.part == NMS_WIDE;
      s_row[tid] = q;
    }
    wide |= __syncthreads_or(odd);
    for (int r0 = 0; r0 < rows; r0 += 64) {
      const int here = rows - r0 < 64 ? rows - r0 : 64;
      const NmsRow me = s_row[r0 + (lane < here ? lane : 0)];
      bool dead = lane >= here;
      const int inlds = K < NMS_KEPT ? K : NMS_KEPT;
      unsigned long long own[64 / NMS_WAVES];   // rows of the block that meet row wave * 4 + u
      if (!wide) {
        int q = wave;
        for (; q + 3 * NMS_WAVES < inlds; q += 4 * NMS_WAVES) {
          bool hit = false;
#pragma unroll
          for (int u = 0; u < 4; ++u) hit |= nms_hits(s_kept[q + u * NMS_WAVES], me, scale);
          dead |= hit;
        }
        for (; q < inlds; q += NMS_WAVES) dead |= nms_hits(s_kept[q], me, scale);
#pragma unroll
        for (int u = 0; u < 64 / NMS_WAVES; ++u) {
          const int i = wave * (64 / NMS_WAVES) + u;
          own[u] = __ballot(nms_hits(s_row[r0 + (i < here ? i : 0)], me, scale));
        }
      } else {
        for (int q = wave; q < inlds; q += NMS_WAVES) dead |= nms_hits_any(s_kept[q], me, iou_threshold);
#pragma unroll 1
        for (int u = 0; u < 64 / NMS_WAVES; ++u) {
          const int i = wave * (64 / NMS_WAVES) + u;
          own[u] = __ballot(nms_hits_any(s_row[r0 + (i < here ? i : 0)], me, iou_threshold));
        }
      }
      for (int q = NMS_KEPT + wave; q < K; q += NMS_WAVES) {
        NmsRow o;
        nms_load_row(o, srt + (int64_t)(kp[q] & 0x7fffffff) * k, coord_start, id_index, iou_threshold);
        if (!by_class) o.id = 0;
        o.seg = ls[q];
        dead |= nms_hits_any(o, me, iou_threshold);
      }
      const unsigned long long dm = __ballot(dead);
      if (lane == 0) {
        if (dm) atomicOr(&s_dead[turn], dm);
#pragma unroll
        for (int u = 0; u < 64 / NMS_WAVES; ++u) s_mask[wave * (64 / NMS_WAVES) + u] = own[u];
      }
      __syncthreads();
      if (wave == 0) {
        unsigned long long gone = s_dead[turn];
        gone = ((unsigned long long)(uint32_t)__builtin_amdgcn_readfirstlane((int)(gone >> 32)) << 32) |
               (uint32_t)__builtin_amdgcn_readfirstlane((int)gone);
        const unsigned long long stay = nms_settle(s_mask[lane] & lt, ~gone, lane);
        if (lane < here) {
          const bool in = (stay >> lane) & 1ull;
          if (in) {
            const int q = K + __popcll(stay & lt);
            if (q < NMS_KEPT) {
              s_kept[q] = me;
            } else {
              kp[q] = me.pos;
              ls[q] = me.seg;
            }
          }
          fl[me.pos & 0x7fffffff] = in && me.pos >= 0;
        }
        if (lane == 0) {
          s_k = K + __popcll(stay);
          s_dead[turn ^ 1] = 0;
        }
      }
      __syncthreads();
      K = __builtin_amdgcn_readfirstlane(s_k);
      turn ^= 1;
    }
  }
}

// The kept rows whose first value is not negative, in sorted order, over the front of the output; max_output_size keeps
// the first so many of them (nms.cc:126-137).
__global__ void __launch_bounds__(256)
k_nms_emit(const int32_t* __restrict__ valid_count, const int32_t* __restrict__ sorted, const uint8_t* __restrict__ flags,
           int32_t* __restrict__ y, int n, int k, int topk, int max_output_size) {
  __shared__ int s_sum[4], s_own[4];
  const int b = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int p0 = blockIdx.x * 256, p = p0 + tid < n ? p0 + tid : n - 1;
  const uint8_t* fl = flags + (int64_t)b * n * 4;
  const int32_t* src = sorted + ((int64_t)b * n + p) * k;
  const uint8_t flag = fl[p];
  int32_t value[ROW_REGS];
  row_request(value, src, k);
  int before = 0;   // flags are bytes of 0 or 1
  for (int w0 = 0; w0 < p0 / 4; w0 += 4 * 256) {
    uint32_t v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int w = w0 + u * 256 + tid;
      v[u] = reinterpret_cast<const uint32_t*>(fl)[w < p0 / 4 ? w : 0];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 4; ++u) before += w0 + u * 256 + tid < p0 / 4 ? __popc(v[u]) : 0;
  }
  if (batch_state(valid_count, b, n) != 0) return;
  const int vc = clamp_vc(valid_count[b], n);
  const int keep = (topk >= 0 && topk < vc) ? topk : vc;
  if (p0 >= keep) return;
  const bool on = p0 + tid < keep && flag != 0;
  for (int d = 32; d >= 1; d >>= 1) before += __shfl_xor(before, d, 64);
  const unsigned long long m = __ballot(on);
  if (lane == 0) {
    s_sum[wave] = before;
    s_own[wave] = __popcll(m);
  }
  __syncthreads();
  int at = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3] + __popcll(m & ((1ull << lane) - 1ull));
  for (int w = 0; w < wave; ++w) at += s_own[w];
  if (!on || (max_output_size > 0 && at >= max_output_size)) return;
  row_store(y + ((int64_t)b * n + at) * k, value, src, k);
}

// ---- scratch of the entry point that allocates nothing (cvmhip_non_max_suppression_static).
// One array per GPU, part of the code object, held until the process ends.  In host code its name is only a
// handle for hipGetSymbolAddress: the device address is looked up once per device, with that device
// current, and only that address is ever passed to a kernel.
constexpr size_t NMS_STATIC_WORDS = (size_t)1 << 19;   // 2 MiB: e.g. one batch of 37 000 rows of 6 values
// a batch takes at least 8 KiB of it, so there are at most 255 batches and as many tallies behind it
constexpr size_t NMS_STATIC_BATCHES = 256;
static_assert((size_t)(BIN_COUNT * 2) * NMS_STATIC_BATCHES >= NMS_STATIC_WORDS, "batches of one row");
static __device__ __align__(256) int32_t g_nms_scratch[NMS_STATIC_WORDS + NMS_STATIC_BATCHES * NMS_TALLY];

constexpr int NMS_MAX_DEVICES = 64;
static std::mutex g_nms_scratch_mu;
static void* g_nms_scratch_ptr[NMS_MAX_DEVICES] = {};

// device address of the current device's copy of the array
static int nms_static_scratch(void** ptr) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= NMS_MAX_DEVICES) {
    set_error("non_max_suppression_static: hipGetDevice: %s (device %d)", hipGetErrorString(e), dev);
    return CVMHIP_ERR_RUNTIME;
  }
  std::lock_guard<std::mutex> lock(g_nms_scratch_mu);
  if (!g_nms_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(g_nms_scratch));
    if (e != hipSuccess || !p) {
      set_error("non_max_suppression_static: hipGetSymbolAddress: %s", hipGetErrorString(e));
      return CVMHIP_ERR_RUNTIME;
    }
    g_nms_scratch_ptr[dev] = p;
  }
  *ptr = g_nms_scratch_ptr[dev];
  return CVMHIP_OK;
}

static int nms_check_args(const int32_t* x, const int32_t* valid_count, const int32_t* y, int batches, int n, int k,
                          int iou_threshold, int coord_start, int score_index, int id_index, int topk) {
  if (!x || !valid_count || !y || x == y || batches < 1 || n < 1 || k < 2 || batches > 65535)
    return arg_error("non_max_suppression");
  if (iou_threshold <= 0) return arg_error("non_max_suppression.iou_threshold must be positive");
  if (coord_start < 0 || coord_start + 4 > k || score_index < 0 || score_index >= k || id_index >= k)
    return arg_error("non_max_suppression indices");
  // 2^24 is the largest dimension the reference's shape check accepts (src/runtime/infer_attr.cc).  The greedy walk compares
  // every row with the kept rows of its class in front of it, and when all candidates (the first top_k in sorted order, or all
  // valid rows) are of one class and stay, one workgroup does that: 5 000 rows take 3 ms, 25 000 0.13 s, 100 000 2.3 s (20
  // classes: 0.2, 0.8 and about 1 ms), growing with the square.  More than 2^18 candidates (some 16 s at worst) are refused
  // rather than launched as a kernel that runs for minutes.
  if (n > (1 << 24)) return arg_error("non_max_suppression: more than 2^24 anchors per batch");
  if (n > (1 << 18) && !(topk >= 0 && topk <= (1 << 18)))
    return arg_error("non_max_suppression: more than 2^18 candidate rows per batch (set top_k to bound the greedy walk)");
  return CVMHIP_OK;
}

// per batch: the words (or list[n] and kept[n]), code[n], sorted[n*k] and either the chunks' and the bins' first
// positions, or rank[n] and the radix sort's two key buffers, two index buffers and digit counts
static size_t nms_rows_bytes(int batches, int n, int k) {
  size_t per = (size_t)n * (3 + (size_t)k);
  if (n >= RADIX_MIN_ROWS) per += (size_t)n * 5 + (size_t)256 * ((n + RADIX_CHUNK - 1) / RADIX_CHUNK);
  else per += (size_t)BIN_COUNT * ((n + BIN_CHUNK - 1) / BIN_CHUNK) + BIN_COUNT + 1;
  return (size_t)batches * per * sizeof(int32_t);
}
// rows of a batch that the walk may see
static int nms_candidates(int n, int topk) { return topk >= 0 && topk < n ? topk : n; }
// overlap masks of a batch's candidates (at most 2^18: nms_check_args)
static int64_t nms_mask_words(int n, int topk) {
  const int most = nms_candidates(n, topk);
  return most < NMS_PAIRS_LEAST ? 0 : (int64_t)(most < (1 << 18) ? most : 1 << 18) * NMS_PAIRS_WORDS;
}

// Validation and launches shared by the two entry points.  `workspace`: nms_rows_bytes(), behind it the tally of every batch and, where
// the caller has room for them, the overlap masks.
static int nms_launch(int32_t* x, const int32_t* valid_count, int32_t* y,
                      int batches, int n, int k, int max_output_size,
                      int iou_threshold, int topk, int coord_start,
                      int score_index, int id_index, int force_suppress,
                      void* workspace, bool has_masks, hipStream_t s) {
  // the words come first: they are 64 bits wide
  unsigned long long* words = reinterpret_cast<unsigned long long*>(workspace);
  int32_t* list = reinterpret_cast<int32_t*>(workspace);   // list and kept take the words' place once the rows are in order
  int32_t* kept = list + (size_t)batches * n;
  int32_t* code = kept + (size_t)batches * n;
  int32_t* sorted = code + (size_t)batches * n;
  int32_t* rank = sorted + (size_t)batches * n * k;   // or the chunks' first positions
  int32_t* tally = reinterpret_cast<int32_t*>(reinterpret_cast<char*>(workspace) + nms_rows_bytes(batches, n, k));
  uint32_t* masks = has_masks ? reinterpret_cast<uint32_t*>(tally) + (size_t)batches * NMS_TALLY : nullptr;
  const dim3 grid((n + 255) / 256, batches);
  int rc;
  if (n >= RADIX_MIN_ROWS) {
    // stable radix sort: two key and two index buffers and the digit counts
    const int nblocks = (n + RADIX_CHUNK - 1) / RADIX_CHUNK;
    uint32_t* keys[2];
    int32_t* idx[2];
    keys[0] = reinterpret_cast<uint32_t*>(rank + (size_t)batches * n);
    keys[1] = keys[0] + (size_t)batches * n;
    idx[0] = reinterpret_cast<int32_t*>(keys[1] + (size_t)batches * n);
    idx[1] = idx[0] + (size_t)batches * n;
    int32_t* hist = idx[1] + (size_t)batches * n;
    rc = CVMHIP_OK;
    for (int pass = 0; pass < 4 && !rc; ++pass) {
      const int in = (pass + 1) & 1, out = pass & 1;   // pass 0 reads the tensor itself
      dim3 rgrid(nblocks, batches);
      k_radix_hist<<<rgrid, RADIX_THREADS, 0, s>>>(x, valid_count, keys[in], hist, n, k, score_index, pass, nblocks, (int64_t)n);
      k_radix_scan<<<batches, 1024, 0, s>>>(valid_count, hist, tally, n, nblocks);
      k_radix_scatter<<<rgrid, RADIX_THREADS, 0, s>>>(x, valid_count, keys[in], idx[in], keys[out], idx[out], hist, rank, n, k,
                                                      score_index, pass, nblocks, (int64_t)n, pass == 3 ? 1 : 0);
      rc = check_launch("nms.radix_sort");
    }
    if (rc) return rc;
    k_nms_scatter<<<grid, 256, 0, s>>>(x, valid_count, rank, code, sorted, y, tally, n, k, topk, id_index);
    rc = check_launch("nms.scatter");
  } else {
    const dim3 cgrid((n + BIN_CHUNK - 1) / BIN_CHUNK, batches);
    int32_t* first = rank + (size_t)batches * cgrid.x * BIN_COUNT;
    k_nms_place<<<cgrid, BIN_CHUNK, 0, s>>>(x, valid_count, rank, first, words, tally, n, k, score_index);
    k_nms_order<<<grid, 256, 0, s>>>(x, valid_count, rank, first, words, code, sorted, y, tally, n, k, topk, id_index);
    rc = check_launch("nms.order");
  }
  if (rc || topk == 0) return rc;
  // the ranks, or positions, have been read: their words hold the keep flags of the sorted positions from here on
  uint8_t* flags = reinterpret_cast<uint8_t*>(rank);
  const int by_class = force_suppress || id_index < 0 ? 0 : 1;
  const int most = nms_candidates(n, topk);
  const int classes = by_class ? NMS_CLASSES : 1;
  if (most < NMS_PAIRS_LEAST) masks = nullptr;
  // A workgroup has a compute unit to itself (100 KiB of LDS): what goes past one round of them is paid by classes that have no pairs
  // for it.  24 564 rows of 21 ids, us for 1, 2, 4, 8 parts: one batch 43.6 37.0 33.3 33.6, two 45.1 38.8 35.9 50.6, four 46.6 41.6
  // 54.5 74.5; four of 5 000 rows (classes too small) 22.1 23.5 30.2 39.8; 400 rows that all meet, four batches: 33.7 29.0 26.1 25.9.
  int parts = 1;
  if (masks) {
    const int most_groups = most >= 8192 ? 512 : 256;
    while (parts < 4 && classes * batches * parts * 2 <= most_groups) parts *= 2;
  }
  k_nms_walk<<<dim3(classes * parts, batches), NMS_THREADS, 0, s>>>(valid_count, sorted, code, list, kept, flags, tally, masks, nms_mask_words(n, topk), n, k,
                                                                   iou_threshold, topk, coord_start, id_index, by_class, parts);
  rc = check_launch("nms.walk");
  if (rc) return rc;
  k_nms_emit<<<dim3((most + 255) / 256, batches), 256, 0, s>>>(valid_count, sorted, flags, y, n, k, topk, max_output_size);
  return check_launch("nms.emit");
}


}  // namespace cvmhip

using namespace cvmhip;

extern "C" {

size_t cvmhip_get_valid_counts_workspace_bytes(int batches, int n) {
  const int nchunks = (n + GVC_CHUNK - 1) / GVC_CHUNK;
  return (size_t)batches * nchunks * sizeof(int32_t);
}

int cvmhip_get_valid_counts(const int32_t* x, int32_t* valid_count, int32_t* y,
                            int batches, int n, int k, int32_t score_threshold,
                            void* workspace, size_t workspace_bytes, void* stream) {
  if (!x || !valid_count || !y || batches < 1 || n < 1 || k < 2 || batches > 65535) return arg_error("get_valid_counts");
  if (!workspace || workspace_bytes < cvmhip_get_valid_counts_workspace_bytes(batches, n))
    return arg_error("get_valid_counts workspace");
  const int nchunks = (n + GVC_CHUNK - 1) / GVC_CHUNK;
  int32_t* counts = reinterpret_cast<int32_t*>(workspace);
  hipStream_t s = as_stream(stream);
  dim3 grid(nchunks, batches);
  if (nchunks <= GVC_OWN_CHUNKS) {
    k_gvc_scatter<true><<<grid, GVC_CHUNK, 0, s>>>(x, counts, valid_count, y, n, k, score_threshold, nchunks);
    return check_launch("get_valid_counts");
  }
  k_gvc_count<<<grid, GVC_CHUNK, 0, s>>>(x, counts, n, k, score_threshold, nchunks);
  int rc = check_launch("get_valid_counts.count");
  if (rc) return rc;
  k_gvc_scatter<false><<<grid, GVC_CHUNK, 0, s>>>(x, counts, valid_count, y, n, k, score_threshold, nchunks);
  return check_launch("get_valid_counts.scatter");
}

size_t cvmhip_nms_topk_workspace_bytes(int batches, int n, int k, int topk) {
  return nms_rows_bytes(batches, n, k) + (size_t)batches * (NMS_TALLY * 4 + (size_t)nms_mask_words(n, topk) * 8);
}
size_t cvmhip_nms_workspace_bytes(int batches, int n, int k) { return cvmhip_nms_topk_workspace_bytes(batches, n, k, -1); }

int cvmhip_non_max_suppression(int32_t* x, const int32_t* valid_count, int32_t* y,
                               int batches, int n, int k, int max_output_size,
                               int iou_threshold, int topk, int coord_start,
                               int score_index, int id_index, int force_suppress,
                               void* workspace, size_t workspace_bytes, void* stream) {
  const int rc = nms_check_args(x, valid_count, y, batches, n, k, iou_threshold, coord_start, score_index, id_index, topk);
  if (rc) return rc;
  if (!workspace || workspace_bytes < cvmhip_nms_topk_workspace_bytes(batches, n, k, topk)) return arg_error("non_max_suppression workspace");
  return nms_launch(x, valid_count, y, batches, n, k, max_output_size, iou_threshold, topk, coord_start, score_index,
                    id_index, force_suppress, workspace, true, as_stream(stream));
}

size_t cvmhip_nms_static_capacity_bytes(void) { return sizeof(int32_t) * NMS_STATIC_WORDS; }

int cvmhip_non_max_suppression_static(int32_t* x, const int32_t* valid_count, int32_t* y,
                                      int batches, int n, int k, int max_output_size,
                                      int iou_threshold, int topk, int coord_start,
                                      int score_index, int id_index, int force_suppress, void* stream) {
  const int rc = nms_check_args(x, valid_count, y, batches, n, k, iou_threshold, coord_start, score_index, id_index, topk);
  if (rc) return rc;
  const size_t need = nms_rows_bytes(batches, n, k);
  if (need > cvmhip_nms_static_capacity_bytes()) {
    set_error("invalid argument: non_max_suppression_static: batches=%d n=%d k=%d needs %zu bytes of scratch, the static "
              "buffer holds %zu; use cvmhip_non_max_suppression with a caller workspace",
              batches, n, k, need, cvmhip_nms_static_capacity_bytes());
    return CVMHIP_ERR_ARG;
  }
  void* scratch = nullptr;
  const int rs = nms_static_scratch(&scratch);
  if (rs) return rs;
  return nms_launch(x, valid_count, y, batches, n, k, max_output_size, iou_threshold, topk, coord_start, score_index,
                    id_index, force_suppress, scratch, false, as_stream(stream));
}

}  // extern "C"
