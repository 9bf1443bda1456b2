// outlier.hip -- outlier scores from a K-nearest-neighbour table (printOutlierScores,
// main.cu:952-1067), a consumer of the join's output.
//
// Per point i of a table with k1 entries per row:
//   dist_sum[i]  = sum over the row of the distances, in entry order, in FP32 (main.cu:966-969)
//   dist_rank[i] = position of i when the points are ordered by dist_sum descending
//   indegree[i]  = number of rows (its own included) in which i appears (main.cu:1011-1020)
//   indeg_rank[i]= position of i when the points are ordered by indegree ascending
// The reference orders with std::sort, which leaves the order of equal values unspecified;
// here equal values are ordered by point id (stable radix sorts over ids 0..N-1), so the ranks
// are deterministic and equal the reference's whenever the values are distinct.
#include <algorithm>

#include "knn_launch.h"

namespace knn {

namespace {

// row sums in entry order; key = bits of the sum arranged so that an ascending unsigned sort
// orders the sums descending (non-negative floats: larger value, larger bits).
// A block takes 256 rows: OUT_E entries of each at a time come in as one coalesced stream and go
// through LDS (odd row stride) to the thread that sums the row.
// COUNT: also counts the in-degrees of the block's entries, by atomics.
constexpr uint32_t OUT_E = 16;
template <bool COUNT>
__global__ __launch_bounds__(256) void k_outlier_rows(const int32_t *__restrict__ ids, const float *__restrict__ dists,
                                                      uint32_t n, uint32_t k1, float *distSum, uint32_t *key,
                                                      uint32_t *val, uint32_t *indeg) {
  __shared__ float tile[256 * (OUT_E + 1)];
  const uint32_t r0 = blockIdx.x * 256u, tid = threadIdx.x;
  const uint32_t rows = n - r0 < 256u ? n - r0 : 256u;
  const uint32_t i = r0 + tid;
  if (COUNT) {
    const int32_t *own = ids + (size_t)r0 * k1;
    for (uint32_t t = tid; t < rows * k1; t += 256) {
      const int32_t id = own[t];
      if (id >= 0 && (uint32_t)id < n) atomicAdd(&indeg[id], 1u);
    }
  }
  const float *src = dists + (size_t)r0 * k1;
  float s = 0.0f;
  for (uint32_t e0 = 0; e0 < k1; e0 += OUT_E) {
    const uint32_t w = k1 - e0 < OUT_E ? k1 - e0 : OUT_E;
    __syncthreads();
    for (uint32_t t = tid; t < rows * w; t += 256) {
      const uint32_t r = t / w, e = t - r * w;
      tile[r * (OUT_E + 1) + e] = src[(size_t)r * k1 + e0 + e];
    }
    __syncthreads();
    if (tid < rows)
      for (uint32_t e = 0; e < w; e++) s += tile[tid * (OUT_E + 1) + e];
  }
  if (i < n) {
    distSum[i] = s;
    const uint32_t b = __float_as_uint(s);
    // -0.0 and +0.0 compare equal; NaN sums (absent entries) sort last
    const uint32_t mag = (s == 0.0f) ? 0u : ((b & 0x80000000u) ? 0u : b);
    key[i] = (s != s) ? 0xffffffffu : 0x7fffffffu - (mag & 0x7fffffffu);
    val[i] = i;
  }
}

// In-degrees.  Counters in global memory take about 28 atomic additions per ns whatever their
// spread (the XCDs' L2s do not share them): 0.6 ms for 17M entries.  With enough entries the ids
// are first dealt into at most DEG_BINS bins of consecutive ids, 16 bits each, and a block per bin
// counts its ids in LDS: the scores of 1M points with 17 entries 0.93 -> 0.37 ms.  With fewer, rows of
// up to 32 are counted by the kernel that sums them (9M points with 4 entries 2.45 -> 2.37 ms, 100k
// with 9 0.307 -> 0.305, 1,000 with 17 0.141 -> 0.137); longer ones by k_deg_atomic, over more
// blocks than they have rows for (1,000 points with 64 entries: 0.160 with the sums, 0.148 so).
constexpr uint32_t ROW_COUNT_K1 = 32;
__global__ void k_deg_atomic(const int32_t *__restrict__ ids, uint64_t m, uint32_t n, uint32_t *indeg) {
  for (uint64_t t = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; t < m; t += (uint64_t)gridDim.x * blockDim.x) {
    const int32_t id = ids[t];
    if (id >= 0 && (uint32_t)id < n) atomicAdd(&indeg[id], 1u);
  }
}

constexpr uint32_t DEG_BINS = 512, DEG_ITEMS = 16;  // bins at most; entries per thread of a scatter block

// binCount[b] += entries of bin b = id >> shift
__global__ __launch_bounds__(256) void k_deg_hist(const int32_t *__restrict__ ids, uint32_t m, uint32_t n,
                                                  uint32_t shift, uint32_t *binCount) {
  __shared__ uint32_t h[DEG_BINS];
  for (uint32_t b = threadIdx.x; b < DEG_BINS; b += 256) h[b] = 0;
  __syncthreads();
  for (uint32_t t0 = blockIdx.x * 2048u + threadIdx.x; t0 < m; t0 += gridDim.x * 2048u) {
    int32_t id[8];
#pragma unroll
    for (uint32_t u = 0; u < 8; u++) id[u] = t0 + 256u * u < m ? ids[t0 + 256u * u] : -1;
#pragma unroll
    for (uint32_t u = 0; u < 8; u++)
      if (id[u] >= 0 && (uint32_t)id[u] < n) atomicAdd(&h[(uint32_t)id[u] >> shift], 1u);
  }
  __syncthreads();
  for (uint32_t b = threadIdx.x; b < DEG_BINS; b += 256)
    if (h[b]) atomicAdd(&binCount[b], h[b]);
}

// one block: binStart = exclusive sums of the counts (DEG_BINS + 1 entries), also the cursors
__global__ __launch_bounds__(DEG_BINS) void k_deg_starts(const uint32_t *binCount, uint32_t *binStart, uint32_t *cursor) {
  __shared__ uint32_t sh[DEG_BINS];
  const uint32_t b = threadIdx.x, c = binCount[b];
  sh[b] = c;
  __syncthreads();
  for (uint32_t o = 1; o < DEG_BINS; o <<= 1) {
    const uint32_t v = b >= o ? sh[b - o] : 0u;
    __syncthreads();
    sh[b] += v;
    __syncthreads();
  }
  binStart[b] = cursor[b] = sh[b] - c;
  if (b == DEG_BINS - 1) binStart[DEG_BINS] = sh[b];
}

// Deals a block's 16384 entries into the bins: ranks from LDS counters, a run per bin reserved at
// the bin's cursor, the entries ordered by bin in LDS so that a run is written by neighbouring
// lanes (scattered 2-byte stores of 4096-entry blocks: 165 us for 17M entries, now 46).
__global__ __launch_bounds__(1024) void k_deg_scatter(const int32_t *__restrict__ ids, uint32_t m, uint32_t n,
                                                      uint32_t shift, uint32_t *cursor, uint16_t *out) {
  __shared__ uint32_t h[DEG_BINS], part[DEG_BINS / 64], order[1024 * DEG_ITEMS];
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  if (tid < DEG_BINS) h[tid] = 0;
  __syncthreads();
  const uint32_t t0 = blockIdx.x * (1024u * DEG_ITEMS) + tid;
  int32_t id[DEG_ITEMS];
  uint32_t rk[DEG_ITEMS];
#pragma unroll
  for (uint32_t u = 0; u < DEG_ITEMS; u++) {
    const uint32_t t = t0 + 1024u * u;
    const int32_t v = t < m ? ids[t] : -1;
    id[u] = v >= 0 && (uint32_t)v < n ? v : -1;
  }
#pragma unroll
  for (uint32_t u = 0; u < DEG_ITEMS; u++) rk[u] = id[u] >= 0 ? atomicAdd(&h[(uint32_t)id[u] >> shift], 1u) : 0u;
  __syncthreads();
  // a bin's first position in the block's order, and its run in the output
  uint32_t c = 0, incl = 0, run = 0;
  if (tid < DEG_BINS) {
    c = incl = h[tid];
    run = c ? atomicAdd(&cursor[tid], c) : 0u;
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t t = (uint32_t)__shfl_up((int)incl, o, 64);
      if ((int)lane >= o) incl += t;
    }
    if (lane == 63) part[tid >> 6] = incl;
  }
  __syncthreads();
  uint32_t total = 0;
  for (uint32_t w = 0; w < DEG_BINS / 64; w++) {
    if (w < tid >> 6) incl += part[w];
    total += part[w];
  }
  if (tid < DEG_BINS) h[tid] = incl - c;
  __syncthreads();
#pragma unroll
  for (uint32_t u = 0; u < DEG_ITEMS; u++)
    if (id[u] >= 0) order[h[(uint32_t)id[u] >> shift] + rk[u]] = (uint32_t)id[u];
  __syncthreads();
  if (tid < DEG_BINS) h[tid] = run - (incl - c);
  __syncthreads();
  for (uint32_t e = tid; e < total; e += 1024) {
    const uint32_t v = order[e];
    out[h[v >> shift] + e] = (uint16_t)(v & ((1u << shift) - 1u));
  }
}

// block b counts bin b's ids; add: onto earlier slabs' counts.  *maxDeg = the largest count.
__global__ __launch_bounds__(1024) void k_deg_count(const uint16_t *__restrict__ binned, const uint32_t *binStart,
                                                    uint32_t n, uint32_t shift, bool add, uint32_t *indeg,
                                                    uint32_t *maxDeg) {
  extern __shared__ uint32_t cnt[];
  const uint32_t size = 1u << shift, i0 = blockIdx.x << shift;
  for (uint32_t e = threadIdx.x; e < size; e += 1024) cnt[e] = 0;
  __syncthreads();
  const uint32_t p1 = binStart[blockIdx.x + 1];
  for (uint32_t p0 = binStart[blockIdx.x] + threadIdx.x; p0 < p1; p0 += 8 * 1024) {
    uint32_t v[8];
#pragma unroll
    for (uint32_t u = 0; u < 8; u++) v[u] = p0 + 1024 * u < p1 ? binned[p0 + 1024 * u] : 0xffffffffu;
#pragma unroll
    for (uint32_t u = 0; u < 8; u++)
      if (v[u] != 0xffffffffu) atomicAdd(&cnt[v[u]], 1u);
  }
  __syncthreads();
  uint32_t mx = 0;
  for (uint32_t e = threadIdx.x; e < size && i0 + e < n; e += 1024) {
    const uint32_t c = cnt[e] + (add ? indeg[i0 + e] : 0u);
    indeg[i0 + e] = c;
    mx = c > mx ? c : mx;
  }
  for (int o = 32; o > 0; o >>= 1) {
    const uint32_t t = (uint32_t)__shfl_xor((int)mx, o, 64);
    mx = t > mx ? t : mx;
  }
  __syncthreads();  // the counters are done with: slot w takes wave w's maximum
  if ((threadIdx.x & 63) == 0) cnt[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t w = 1; w < 16; w++) mx = cnt[w] > mx ? cnt[w] : mx;
    atomicMax(maxDeg, mx);
  }
}

__global__ void k_indeg_keys(const uint32_t *indeg, uint32_t n, uint32_t *key, uint32_t *val) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  key[i] = indeg[i];
  val[i] = i;
}

// rank[val[p]] = p for the sorted order
__global__ void k_scatter_rank(const uint32_t *val, uint32_t n, uint32_t *rank) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  rank[val[p]] = p;
}

}  // namespace

// The largest number of entries dealt at once: 64 MB of 16-bit ids.
constexpr uint64_t DEG_SLAB = 1ull << 25;
// Bins of 2^shift ids, at least 1024 so that small tables keep few bins and at most 16384 (64 KB
// of LDS); from 4M entries on, where the counters' atomics take 0.14 ms (below, the four extra
// launches cost what they save: 100k points with 9 entries 0.30 ms either way), and to 8M points.
OutlierPlan outlier_plan(uint32_t n, uint32_t k1) {
  OutlierPlan p{};
  const uint64_t m = (uint64_t)n * k1;
  uint32_t shift = 10;
  while (shift < 14 && ((uint64_t)n >> shift) >= DEG_BINS) shift++;
  if (m < (1ull << 22) || k1 > DEG_SLAB || ((uint64_t)n >> shift) >= DEG_BINS) return p;
  p.shift = shift;
  p.slabRows = (uint32_t)std::min<uint64_t>(n, DEG_SLAB / k1);
  p.words = ((size_t)p.slabRows * k1 + 1) / 2 + 3 * DEG_BINS + 64;
  return p;
}

hipError_t outlier_scores(const int32_t *ids, const float *dists, uint32_t n, uint32_t k1, float *distSum,
                          uint32_t *distRank, uint32_t *indeg, uint32_t *indegRank, uint32_t *keys,
                          uint32_t *vals, uint32_t *keysTmp, uint32_t *valsTmp, uint32_t *scratch,
                          const OutlierPlan &p, uint32_t *bins, uint32_t *pinnedWord, hipStream_t s) {
  if (!n) return hipSuccess;
  const uint32_t g = (n + 255) / 256;
  int degBits = 32;
  if (p.shift) {
    uint32_t *count = bins, *start = bins + DEG_BINS, *cursor = start + DEG_BINS + 1, *maxDeg = cursor + DEG_BINS;
    uint16_t *binned = reinterpret_cast<uint16_t *>(bins + 3 * DEG_BINS + 64);
    const uint32_t nb = ((n - 1u) >> p.shift) + 1u;
    fill_u32(maxDeg, 0u, 1, s);
    for (uint32_t r0 = 0; r0 < n; r0 += p.slabRows) {
      const uint32_t m = std::min(p.slabRows, n - r0) * k1;
      const int32_t *sl = ids + (size_t)r0 * k1;
      fill_u32(count, 0u, DEG_BINS, s);
      k_deg_hist<<<std::min<uint32_t>((m + 2047) / 2048, 1024u), 256, 0, s>>>(sl, m, n, p.shift, count);
      k_deg_starts<<<1, DEG_BINS, 0, s>>>(count, start, cursor);
      k_deg_scatter<<<(m + 1024 * DEG_ITEMS - 1) / (1024 * DEG_ITEMS), 1024, 0, s>>>(sl, m, n, p.shift, cursor, binned);
      k_deg_count<<<nb, 1024, sizeof(uint32_t) << p.shift, s>>>(binned, start, n, p.shift, r0 != 0, indeg, maxDeg);
    }
    const hipError_t e = hipMemcpyAsync(pinnedWord, maxDeg, sizeof(uint32_t), hipMemcpyDeviceToHost, s);
    if (e != hipSuccess) return e;
  } else {
    fill_u32(indeg, 0u, n, s);
    const uint64_t m = (uint64_t)n * k1;
    if (k1 > ROW_COUNT_K1) k_deg_atomic<<<(uint32_t)std::min<uint64_t>((m + 255) / 256, 8192u), 256, 0, s>>>(ids, m, n, indeg);
  }
  auto rows = !p.shift && k1 <= ROW_COUNT_K1 ? k_outlier_rows<true> : k_outlier_rows<false>;
  rows<<<g, 256, 0, s>>>(ids, dists, n, k1, distSum, keys, vals, indeg);
  radix_sort_pairs_u32(keys, vals, keysTmp, valsTmp, n, 32, scratch, s);
  k_scatter_rank<<<g, 256, 0, s>>>(vals, n, distRank);
  k_indeg_keys<<<g, 256, 0, s>>>(indeg, n, keys, vals);
  if (p.shift) {
    const hipError_t e = hipStreamSynchronize(s);
    if (e != hipSuccess) return e;
    degBits = 1;  // the keys' digits: one 8-bit pass instead of four for most tables
    while (degBits < 32 && (*pinnedWord >> degBits)) degBits++;
  }
  radix_sort_pairs_u32(keys, vals, keysTmp, valsTmp, n, degBits, scratch, s);
  k_scatter_rank<<<g, 256, 0, s>>>(vals, n, indegRank);
  return hipSuccess;
}

}  // namespace knn
