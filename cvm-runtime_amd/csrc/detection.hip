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
// batch total are filled with -1.
__global__ void __launch_bounds__(GVC_CHUNK)
k_gvc_scatter(const int32_t* __restrict__ x, const int32_t* __restrict__ counts, int32_t* __restrict__ valid_count,
              int32_t* __restrict__ y, int n, int k, int32_t thr, int nchunks) {
  __shared__ int wsum[GVC_CHUNK / 64];
  __shared__ int s_bef[GVC_CHUNK / 64], s_tot[GVC_CHUNK / 64];
  __shared__ int s_before, s_total;
  const int b = blockIdx.y, chunk = blockIdx.x;
  {
    // the counts are summed by all threads (one thread walking a hundred of them is a chain of a hundred loads)
    int before = 0, total = 0;
    for (int c = threadIdx.x; c < nchunks; c += GVC_CHUNK) {
      const int v = counts[b * nchunks + c];
      before += c < chunk ? v : 0;
      total += v;
    }
    for (int d = 32; d >= 1; d >>= 1) {
      before += __shfl_xor(before, d, 64);
      total += __shfl_xor(total, d, 64);
    }
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
  const int row = chunk * GVC_CHUNK + threadIdx.x;
  const int32_t* src = x + ((int64_t)b * n + row) * k;
  const bool keep = row < n && src[1] > thr;
  const unsigned long long m = __ballot(keep);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int in_wave = __popcll(m & ((1ull << lane) - 1ull));
  if (lane == 0) wsum[wv] = __popcll(m);
  __syncthreads();
  int pos = s_before + in_wave;
  for (int i = 0; i < wv; ++i) pos += wsum[i];
  int32_t* yb = y + (int64_t)b * n * k;
  if (keep)
    for (int c = 0; c < k; ++c) yb[(int64_t)pos * k + c] = src[c];
  if (row < n && row >= s_total)
    for (int c = 0; c < k; ++c) yb[(int64_t)row * k + c] = -1;
}

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

constexpr int NMS_CLASSES = 64;   // workgroups the candidate rows of a batch are dealt to by id

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
// 9 000 rows with 8-bit scores: 11 us against 27 us for counting all pairs and moving the rows, and 75 us for the
// twelve launches of the radix sort below.  Rows that share one bin (all scores equal) cost n^2 comparisons spread
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
            int32_t* __restrict__ first, unsigned long long* __restrict__ words, int n, int k, int score_index) {
  __shared__ int s_before[BIN_COUNT], s_rest[BIN_COUNT], s_sum[BIN_COUNT / 64];   // rows of earlier chunks, of the others
  const int b = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (batch_state(valid_count, b, n) != 0) return;
  const int vc = clamp_vc(valid_count[b], n);
  const int chunk = blockIdx.x, chunks = (vc + BIN_CHUNK - 1) / BIN_CHUNK;
  if (chunk >= chunks) return;
  const int32_t* xb = x + (int64_t)b * n * k + score_index;
  s_before[tid] = 0;
  s_rest[tid] = 0;
  const int row = chunk * BIN_CHUNK + tid;
  const int32_t score = xb[(int64_t)(row < vc ? row : vc - 1) * k];
  __syncthreads();
  for (int c0 = 0; c0 < chunks; c0 += 8) {
    int32_t v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = (c0 + u) * BIN_CHUNK + tid;
      v[u] = xb[(int64_t)(i < vc ? i : vc - 1) * k];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if ((c0 + u) * BIN_CHUNK + tid < vc) atomicAdd(c0 + u < chunk ? &s_before[score_bin(v[u])] : &s_rest[score_bin(v[u])], 1);
  }
  __syncthreads();
  const int before = s_before[tid], total = before + s_rest[tid];
  int run = total;
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(run, d, 64);
    if (lane >= d) run += o;
  }
  if (lane == 63) s_sum[wave] = run;
  __syncthreads();
  int start = run - total;
  for (int w = 0; w < wave; ++w) start += s_sum[w];
  if (chunk == 0) first[(int64_t)b * (BIN_COUNT + 1) + tid] = start;
  if (chunk == 0 && tid == 0) first[(int64_t)b * (BIN_COUNT + 1) + BIN_COUNT] = vc;
  mine[((int64_t)b * gridDim.x + chunk) * BIN_COUNT + tid] = start + before;
  s_before[tid] = start + before;
  __syncthreads();
  if (row < vc) words[(int64_t)b * n + atomicAdd(&s_before[score_bin(score)], 1)] = score_word(score, row);
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
k_radix_scan(const int32_t* __restrict__ valid_count, int32_t* __restrict__ hist, int n, int nblocks) {
  __shared__ int s_sum[1024];
  const int b = blockIdx.x, tid = threadIdx.x;
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
__device__ __forceinline__ void nms_move_row(int32_t* __restrict__ x, int32_t* __restrict__ code, int32_t* __restrict__ sorted,
                                             int b, int n, int k, int i, int r, int topk, int id_index) {
  int32_t* xrow = x + ((int64_t)b * n + i) * k;
  if (topk > 0 && r >= topk) {  // never looked at again
    for (int c = 0; c < k; ++c) xrow[c] = -1;
    return;
  }
  code[(int64_t)b * n + r] = (id_index >= 0 ? xrow[id_index] & (NMS_CLASSES - 1) : 0) | (xrow[0] < 0 ? 256 : 0);
  int32_t* dst = sorted + ((int64_t)b * n + r) * k;
  for (int c = 0; c < k; ++c) dst[c] = xrow[c];
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
              int32_t* __restrict__ code, int32_t* __restrict__ sorted, int32_t* __restrict__ y, int n, int k,
              int topk, int id_index) {
  const int b = blockIdx.y;
  const int state = batch_state(valid_count, b, n);
  if (state == 2) return;
  nms_clear_rows(y, b, n, k, blockIdx.x * 256);
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (state == 1 || i >= clamp_vc(valid_count[b], n)) return;
  nms_move_row(x, code, sorted, b, n, k, i, rank[(int64_t)b * n + i], topk, id_index);
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
            int32_t* __restrict__ sorted, int32_t* __restrict__ y, int n, int k, int topk, int id_index) {
  __shared__ unsigned long long s_word[BIN_STAGE];
  const int b = blockIdx.y, p0 = blockIdx.x * 256, tid = threadIdx.x;
  const int state = batch_state(valid_count, b, n);
  if (state == 2) return;
  nms_clear_rows(y, b, n, k, p0);
  if (state == 1) return;
  const int vc = clamp_vc(valid_count[b], n);
  if (p0 >= vc) return;
  const unsigned long long* wb = words + (int64_t)b * n;
  const int32_t* fb = first + (int64_t)b * (BIN_COUNT + 1);
  const bool live = p0 + tid < vc;
  const int last = p0 + 255 < vc ? p0 + 255 : vc - 1;
  const unsigned long long me = wb[live ? p0 + tid : last], head = wb[p0], tail = wb[last];
  const int32_t score = (int32_t)((uint32_t)(me >> 32) ^ 0x80000000u);
  const int bin = score_bin(score), row = (int)~(uint32_t)me;
  int lo = fb[bin], hi = fb[bin + 1];
  const int from = fb[score_bin((int32_t)((uint32_t)(head >> 32) ^ 0x80000000u))];
  const int to = fb[score_bin((int32_t)((uint32_t)(tail >> 32) ^ 0x80000000u)) + 1];
  const bool past = topk > 0 && lo >= topk;   // every row of this bin is past top_k: which rank it has is of no interest
  if (!past && hi - lo > 128 && score < BIN_EXACT && ~score < BIN_EXACT) {
    const int chunk = row / BIN_CHUNK;
    const int32_t* m = mine + ((int64_t)b * ((n + BIN_CHUNK - 1) / BIN_CHUNK) + chunk) * BIN_COUNT + bin;
    lo = m[0];
    if ((chunk + 1) * BIN_CHUNK < vc) hi = m[BIN_COUNT];
  }
  int r = lo;
  if (to - from <= BIN_STAGE) {
    for (int t = from + tid; t < to; t += 256) s_word[t - from] = wb[t];
    __syncthreads();
    if (!past) r += nms_count_above(s_word, lo - from, hi - from, me);
  } else if (!past) {
    r += nms_count_above(wb, lo, hi, me);
  }
  if (live) nms_move_row(x, code, sorted, b, n, k, row, r, topk, id_index);
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
// 9 000 of them valid, 21 ids: 22.5 ms in the row-by-row walk of one workgroup, 29 us here; the first 400 rows: 6 us.
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
  q.x1 = row[coord_start];
  q.y1 = row[coord_start + 1];
  q.x2 = row[coord_start + 2];
  q.y2 = row[coord_start + 3];
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

__global__ void __launch_bounds__(NMS_THREADS)
k_nms_walk(const int32_t* __restrict__ valid_count, const int32_t* __restrict__ sorted, const int32_t* __restrict__ code,
           int32_t* __restrict__ list, int32_t* __restrict__ kept, uint8_t* __restrict__ flags, int n, int k,
           int iou_threshold, int topk, int coord_start, int id_index, int by_class) {
  __shared__ NmsRow s_row[NMS_WINDOW];
  __shared__ NmsRow s_kept[NMS_KEPT];
  __shared__ unsigned long long s_mask[64], s_dead[2];
  __shared__ int s_count[NMS_WAVES][3], s_k;
  const int b = blockIdx.y, cls = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (batch_state(valid_count, b, n) != 0) return;
  const int vc = clamp_vc(valid_count[b], n);
  const int keep = (topk >= 0 && topk < vc) ? topk : vc;
  const int32_t* srt = sorted + (int64_t)b * n * k;
  const int32_t* cd = code + (int64_t)b * n;
  uint8_t* fl = flags + (int64_t)b * n * 4;
  const unsigned long long lt = (1ull << lane) - 1ull;

  // this workgroup's rows in sorted order: every wavefront counts its own stretch of the codes, then lists it
  const int per = ((keep + NMS_WAVES - 1) / NMS_WAVES + 63) & ~63;
  const int lo = wave * per, hi = lo + per < keep ? lo + per : keep;
  int mine = 0, lower = 0, neg = 0;
  for (int p0 = lo; p0 < hi; p0 += 256) {
    int c[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int p = p0 + u * 64 + lane;
      c[u] = cd[p < hi ? p : hi - 1];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool in = p0 + u * 64 + lane < hi;
      mine += __popcll(__ballot(in && (!by_class || (c[u] & 255) == cls)));
      lower += __popcll(__ballot(in && by_class && (c[u] & 255) < cls));
      neg += __popcll(__ballot(in && c[u] >= 256));
    }
  }
  if (lane == 0) {
    s_count[wave][0] = mine;
    s_count[wave][1] = lower;
    s_count[wave][2] = neg;
  }
  if (tid < 2) s_dead[tid] = 0;
  __syncthreads();
  int total = 0, base = 0, at = 0, seg = 0, cuts = 0;
#pragma unroll
  for (int w = 0; w < NMS_WAVES; ++w) {
    total += s_count[w][0];
    base += s_count[w][1];
    cuts += s_count[w][2];
    at += w < wave ? s_count[w][0] : 0;
    seg += w < wave ? s_count[w][2] : 0;
  }
  total = __builtin_amdgcn_readfirstlane(total);
  if (total == 0) return;
  // rows past the first window, and later the kept rows past NMS_KEPT, live in memory at this class's own stretch
  int32_t* ls = list + (int64_t)b * n + base;
  // (list: position of row t, kept: its seg; once row t is staged, kept row q <= t goes to the same slots)
  int32_t* kp = kept + (int64_t)b * n + base;
  for (int p0 = lo; p0 < hi; p0 += 256) {
    int c[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int p = p0 + u * 64 + lane;
      c[u] = cd[p < hi ? p : hi - 1];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int p = p0 + u * 64 + lane;
      const bool own = p < hi && (!by_class || (c[u] & 255) == cls), ng = p < hi && c[u] >= 256;
      const unsigned long long om = __ballot(own), nm = __ballot(ng);
      if (own) {
        const int t = at + __popcll(om & lt), sg = seg + __popcll(nm & lt) + (ng ? 1 : 0);
        const int word = p | (ng ? (int)0x80000000u : 0);
        if (t < NMS_WINDOW) {
          s_row[t].pos = word;
          s_row[t].seg = sg;
        } else {
          ls[t] = word;
          kp[t] = sg;
        }
      }
      at += __popcll(om);
      seg += __popcll(nm);
    }
  }
  __syncthreads();

  int K = 0, turn = 0, wide = cuts != 0;
  const uint32_t scale = 100u + (uint32_t)iou_threshold;
  for (int w0 = 0; w0 < total; w0 += NMS_WINDOW) {
    const int rows = total - w0 < NMS_WINDOW ? total - w0 : NMS_WINDOW;
    int odd = 0;
    if (tid < rows) {
      NmsRow q;
      q.pos = w0 ? ls[w0 + tid] : s_row[tid].pos;
      q.seg = w0 ? kp[w0 + tid] : s_row[tid].seg;
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
        // rows in front of this lane's row that would remove it (overlap is symmetric).  A row stays when none of them
        // is kept or still open, and goes when one of them is kept: a few rounds settle the block (the first open row
        // is settled in every round), where a walk takes a step per overlapping row.
        const unsigned long long m = s_mask[lane] & lt;
        unsigned long long gone = s_dead[turn];
        gone = ((unsigned long long)(uint32_t)__builtin_amdgcn_readfirstlane((int)(gone >> 32)) << 32) |
               (uint32_t)__builtin_amdgcn_readfirstlane((int)gone);
        unsigned long long open = ~gone, stay = 0;
        while (open) {
          const bool mineopen = (open >> lane) & 1ull;
          const unsigned long long now = __ballot(mineopen && !(m & (stay | open)));
          stay |= now;
          open &= ~(now | __ballot(mineopen && (m & stay)));
        }
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
  if (batch_state(valid_count, b, n) != 0) return;
  const int vc = clamp_vc(valid_count[b], n);
  const int keep = (topk >= 0 && topk < vc) ? topk : vc;
  const int p0 = blockIdx.x * 256;
  if (p0 >= keep) return;
  const uint8_t* fl = flags + (int64_t)b * n * 4;
  const bool on = p0 + tid < keep && fl[p0 + tid] != 0;
  int before = 0;   // flags are bytes of 0 or 1
  for (int w = tid; w < p0 / 4; w += 256) before += __popc(reinterpret_cast<const uint32_t*>(fl)[w]);
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
  const int32_t* src = sorted + ((int64_t)b * n + p0 + tid) * k;
  int32_t* dst = y + ((int64_t)b * n + at) * k;
  for (int c = 0; c < k; ++c) dst[c] = src[c];
}

// ---- scratch of the entry point that allocates nothing (cvmhip_non_max_suppression_static).
// One array per GPU, part of the code object, held until the process ends.  In host code its name is only a
// handle for hipGetSymbolAddress: the device address is looked up once per device, with that device
// current, and only that address is ever passed to a kernel.
constexpr size_t NMS_STATIC_WORDS = (size_t)1 << 19;   // 2 MiB: e.g. one batch of 37 000 rows of 6 values
static __device__ __align__(256) int32_t g_nms_scratch[NMS_STATIC_WORDS];

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

// Validation and launches shared by the two entry points; `workspace` holds cvmhip_nms_workspace_bytes() bytes.
static int nms_launch(int32_t* x, const int32_t* valid_count, int32_t* y,
                      int batches, int n, int k, int max_output_size,
                      int iou_threshold, int topk, int coord_start,
                      int score_index, int id_index, int force_suppress,
                      void* workspace, hipStream_t s) {
  // the words come first: they are 64 bits wide
  unsigned long long* words = reinterpret_cast<unsigned long long*>(workspace);
  int32_t* list = reinterpret_cast<int32_t*>(workspace);   // list and kept take the words' place once the rows are in order
  int32_t* kept = list + (size_t)batches * n;
  int32_t* code = kept + (size_t)batches * n;
  int32_t* sorted = code + (size_t)batches * n;
  int32_t* rank = sorted + (size_t)batches * n * k;   // or the chunks' first positions
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
      k_radix_scan<<<batches, 1024, 0, s>>>(valid_count, hist, n, nblocks);
      k_radix_scatter<<<rgrid, RADIX_THREADS, 0, s>>>(x, valid_count, keys[in], idx[in], keys[out], idx[out], hist, rank, n, k,
                                                      score_index, pass, nblocks, (int64_t)n, pass == 3 ? 1 : 0);
      rc = check_launch("nms.radix_sort");
    }
    if (rc) return rc;
    k_nms_scatter<<<grid, 256, 0, s>>>(x, valid_count, rank, code, sorted, y, n, k, topk, id_index);
    rc = check_launch("nms.scatter");
  } else {
    const dim3 cgrid((n + BIN_CHUNK - 1) / BIN_CHUNK, batches);
    int32_t* first = rank + (size_t)batches * cgrid.x * BIN_COUNT;
    k_nms_place<<<cgrid, BIN_CHUNK, 0, s>>>(x, valid_count, rank, first, words, n, k, score_index);
    k_nms_order<<<grid, 256, 0, s>>>(x, valid_count, rank, first, words, code, sorted, y, n, k, topk, id_index);
    rc = check_launch("nms.order");
  }
  if (rc || topk == 0) return rc;
  // the ranks, or positions, have been read: their words hold the keep flags of the sorted positions from here on
  uint8_t* flags = reinterpret_cast<uint8_t*>(rank);
  const int by_class = force_suppress || id_index < 0 ? 0 : 1;
  k_nms_walk<<<dim3(by_class ? NMS_CLASSES : 1, batches), NMS_THREADS, 0, s>>>(valid_count, sorted, code, list, kept, flags, n, k,
                                                                              iou_threshold, topk, coord_start, id_index, by_class);
  rc = check_launch("nms.walk");
  if (rc) return rc;
  const int most = topk > 0 && topk < n ? topk : n;
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
  k_gvc_count<<<grid, GVC_CHUNK, 0, s>>>(x, counts, n, k, score_threshold, nchunks);
  int rc = check_launch("get_valid_counts.count");
  if (rc) return rc;
  k_gvc_scatter<<<grid, GVC_CHUNK, 0, s>>>(x, counts, valid_count, y, n, k, score_threshold, nchunks);
  return check_launch("get_valid_counts.scatter");
}

// per batch: the words (or list[n] and kept[n]), code[n], sorted[n*k] and either the chunks' and the bins' first
// positions, or rank[n] and the radix sort's two key buffers, two index buffers and digit counts
size_t cvmhip_nms_workspace_bytes(int batches, int n, int k) {
  size_t per = (size_t)n * (3 + (size_t)k);
  if (n >= RADIX_MIN_ROWS) per += (size_t)n * 5 + (size_t)256 * ((n + RADIX_CHUNK - 1) / RADIX_CHUNK);
  else per += (size_t)BIN_COUNT * ((n + BIN_CHUNK - 1) / BIN_CHUNK) + BIN_COUNT + 1;
  return (size_t)batches * per * sizeof(int32_t);
}

int cvmhip_non_max_suppression(int32_t* x, const int32_t* valid_count, int32_t* y,
                               int batches, int n, int k, int max_output_size,
                               int iou_threshold, int topk, int coord_start,
                               int score_index, int id_index, int force_suppress,
                               void* workspace, size_t workspace_bytes, void* stream) {
  const int rc = nms_check_args(x, valid_count, y, batches, n, k, iou_threshold, coord_start, score_index, id_index, topk);
  if (rc) return rc;
  if (!workspace || workspace_bytes < cvmhip_nms_workspace_bytes(batches, n, k)) return arg_error("non_max_suppression workspace");
  return nms_launch(x, valid_count, y, batches, n, k, max_output_size, iou_threshold, topk, coord_start, score_index,
                    id_index, force_suppress, workspace, as_stream(stream));
}

size_t cvmhip_nms_static_capacity_bytes(void) { return sizeof(int32_t) * NMS_STATIC_WORDS; }

int cvmhip_non_max_suppression_static(int32_t* x, const int32_t* valid_count, int32_t* y,
                                      int batches, int n, int k, int max_output_size,
                                      int iou_threshold, int topk, int coord_start,
                                      int score_index, int id_index, int force_suppress, void* stream) {
  const int rc = nms_check_args(x, valid_count, y, batches, n, k, iou_threshold, coord_start, score_index, id_index, topk);
  if (rc) return rc;
  const size_t need = cvmhip_nms_workspace_bytes(batches, n, k);
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
                    id_index, force_suppress, scratch, as_stream(stream));
}

}  // extern "C"
