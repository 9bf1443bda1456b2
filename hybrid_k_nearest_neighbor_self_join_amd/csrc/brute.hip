// brute.hip -- exact top-(K+1) of a list of queries against every point, without the index.
//
// Counterpart of the reference's no-selectivity path: distanceTableNDBruteForce
// (GPU.cu:1903-2930) with kernelNDBruteForce (kernel.cu:902-975), which emits every
// (query, point, distance) triple into the pair buffer and sorts it, and the criterion
// checkIndexSelectivity (main.cu:2687-2716) that would select it (both unused by the
// reference's main loop).  Here no pair is stored: each query keeps its K+1 best in LDS.
//
// Ranking is that of the range kernels: FP64 key = sum_j ((double)c_j - (double)q_j)^2 (dims
// in the reordered order, no FMA), ties by point id; the reported distance is sqrt of the
// input-type sum sum_j (c_j - q_j)^2.  A row is therefore bit-identical to the one the range
// kernels write for the same query.
//
// k_brute_sample (up to BR_SAMPLE_NQ queries split over chunks): an upper bound of each query's
//   (K+1)-th key, the (K+1)-th smallest of a sample of the points.
// k_brute_partial: one wave per (tile of up to 4 queries, chunk of points); lane = point,
//   64 points per round, each point's key computed for every query of the tile.  Candidates
//   below the query's current (K+1)-th (key, id) are appended to an LDS buffer through a
//   ballot; a full buffer is bitonic-sorted and merged into the sorted best list by rank
//   (each element's output position = own index + elements of the other list before it).
//   With one chunk the kernel writes the rows; otherwise what each chunk holds (up to its K+1
//   best) is appended to the query's partial list.
// k_brute_merge: one wave per query streams its partial list through the same collector
//   and writes the row.
// Without the bound every chunk fills and merges K+1 candidates before its threshold means
// anything, and the merge streams (K+1) entries per chunk: a tail of 1 query over 1.3M 2-D points
// at K = 100 took 0.75 ms and takes 0.15 (sample 21 us, scan 25, merge 109); joins of 5M 4-D
// points at K = 32 with tails of 245 and 128 queries 22.4 -> 21.5 and 22.3 -> 21.6 ms.
#include <algorithm>
#include <type_traits>

#include "knn_collect.h"
#include "knn_launch.h"

namespace knn {

namespace {

constexpr uint32_t BR_QW = 4;  // queries per wave in k_brute_partial (upper bound)
constexpr uint32_t BR_SAMPLE_NQ = 4096;

template <int D, typename T>
__device__ __forceinline__ double br_key(const T *c, const T *q) {
  double s = 0.0;
#pragma unroll
  for (int j = 0; j < D; j++) {
    const double dx = (double)c[j] - (double)q[j];
    const double t = dx * dx;
    s = s + t;
  }
  return s;
}

template <int D, typename T>
__device__ __forceinline__ T br_dist_sq(const T *c, const T *q) {
  T s = (T)0;
#pragma unroll
  for (int j = 0; j < D; j++) {
    const T df = c[j] - q[j];
    const T t = df * df;
    s = s + t;
  }
  return s;
}

// writes query q's row from a finished collector (entries past nb, possible only when fewer
// than k1 points exist, are left as id -1 / distance 0)
template <typename T, int D>
__device__ void br_write_row(const BruteArgs &a, const Collector &c, uint32_t q, uint32_t lane) {
  const T *x = static_cast<const T *>(a.x);
  T qc[D];
#pragma unroll
  for (int j = 0; j < D; j++) qc[j] = x[(size_t)j * a.n + q];
  const size_t row = (size_t)q * a.k1;
  T *od = static_cast<T *>(a.outDists);
  for (uint32_t e = lane; e < a.k1; e += 64) {
    if (e < c.nb) {
      const uint32_t id = c.best_id(e);
      T cc[D];
#pragma unroll
      for (int j = 0; j < D; j++) cc[j] = x[(size_t)j * a.n + id];
      a.outIds[row + e] = (int32_t)id;
      od[row + e] = sqrt(br_dist_sq<D, T>(cc, qc));
    } else {
      a.outIds[row + e] = -1;
      od[row + e] = (T)0;
    }
  }
  if (lane == 0 && a.failed) a.failed[q] = 0;
}

// One block per query: bound[qi] >= the (K+1)-th smallest key over a.sample points, runs of 64
// spread evenly over all of them, and so of the whole set's.  Radix selection (11 + 11 + 10 bits)
// on the bits of the keys rounded to float, which order as the keys do; the selected value's
// upper neighbour is above every key that rounds to it.  NaN keys are not counted; with fewer
// than K+1 left the bound is infinite.
template <typename T, int D>
__global__ __launch_bounds__(1024) void k_brute_sample(BruteArgs a) {
  __shared__ uint32_t hist[2048], part[16], sel[2];
  const uint32_t tid = threadIdx.x, lane = tid & 63, qi = blockIdx.x;
  const T *x = static_cast<const T *>(a.x);
  const uint32_t q = a.queries ? a.queries[qi] : qi;
  T qc[D];
#pragma unroll
  for (int j = 0; j < D; j++) qc[j] = x[(size_t)j * a.n + q];
  const uint32_t runs = a.sample / 64;  // a.sample <= n / 4: the runs do not overlap
  const uint64_t step = a.n / runs;
  uint32_t prefix = 0, rank = a.k1;  // the rank-th (from 1) smallest of those with this prefix
  for (int pass = 0; pass < 3; pass++) {
    const uint32_t shift = pass == 0 ? 21u : (pass == 1 ? 10u : 0u), nb = pass == 2 ? 1024u : 2048u;
    for (uint32_t e = tid; e < 2048; e += 1024) hist[e] = 0;
    __syncthreads();
#pragma unroll 4
    for (uint32_t r = tid >> 6; r < runs; r += 16) {
      const uint32_t p = (uint32_t)(r * step) + lane;
      T c[D];
#pragma unroll
      for (int j = 0; j < D; j++) c[j] = x[(size_t)j * a.n + p];
      const float f = (float)br_key<D, T>(c, qc);
      const uint32_t b = __float_as_uint(f);
      bool in = f == f && (pass == 0 || (b >> (pass == 1 ? 21 : 10)) == prefix);
      const uint32_t dig = (b >> shift) & (nb - 1u);
      // most lanes of a run often share a digit: one add for those of the first lane's
      const uint64_t m = __ballot(in);
      if (m) {
        const int first = __ffsll((long long)m) - 1;
        const bool same = in && dig == (uint32_t)__shfl((int)dig, first, 64);
        const uint64_t ms = __ballot(same);
        if ((int)lane == first) atomicAdd(&hist[dig], (uint32_t)__popcll(ms));
        if (in && !same) atomicAdd(&hist[dig], 1u);
      }
    }
    __syncthreads();
    // the digit that holds the rank: two counters per thread, scanned over the block
    const uint32_t h0 = hist[2 * tid], h1 = hist[2 * tid + 1];
    uint32_t incl = h0 + h1;
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t t = (uint32_t)__shfl_up((int)incl, o, 64);
      if ((int)lane >= o) incl += t;
    }
    if (lane == 63) part[tid >> 6] = incl;
    if (tid == 0) sel[0] = 0xffffffffu;
    __syncthreads();
    uint32_t before = incl - h0 - h1;
    for (uint32_t w = 0; w < tid >> 6; w++) before += part[w];
    if (before < rank && rank <= before + h0 + h1) {
      const bool second = rank > before + h0;
      sel[0] = 2 * tid + (second ? 1u : 0u);
      sel[1] = rank - before - (second ? h0 : 0u);
    }
    __syncthreads();
    const uint32_t dig = sel[0];
    rank = sel[1];
    if (dig == 0xffffffffu) {  // fewer than K+1 ordered keys
      if (tid == 0) a.bound[qi] = __builtin_inf();
      return;
    }
    prefix = pass == 0 ? dig : (pass == 1 ? (prefix << 11) | dig : (prefix << 10) | dig);
    __syncthreads();
  }
  if (tid == 0) a.bound[qi] = (double)__uint_as_float(prefix < 0x7f800000u ? prefix + 1u : prefix);
}

// U: rounds of points loaded together.  Several for a tail of few queries, whose waves wait for
// memory; one for a whole join, whose waves are many and bound by issue (28,903 uniform 4-D points,
// K=8: 1.25 ms, with four rounds 1.35).
template <typename T, int D, uint32_t U>
__global__ __launch_bounds__(64) void k_brute_partial(BruteArgs a) {
  extern __shared__ __align__(16) unsigned char br_lds[];
  const uint32_t lane = threadIdx.x;
  // consecutive blocks share a chunk of points, which then comes from the L2 for all but one
  const uint32_t tiles = (a.nq + a.qw - 1) / a.qw;
  const uint32_t chunk = blockIdx.x / tiles;
  const uint32_t tile = blockIdx.x - chunk * tiles;
  const uint32_t q0 = tile * a.qw;
  const uint32_t qw = (a.nq - q0) < a.qw ? (a.nq - q0) : a.qw;
  const T *x = static_cast<const T *>(a.x);

  Collector col[BR_QW];
  T qc[BR_QW][D];
  uint32_t qid[BR_QW];
  // float input: the FP32 sum s = sum_j (c_j - q_j)^2 is within 2^-19 of the FP64 key
  // relative, so a point whose key can reach the threshold tk has s <= tk (1 + 2^-16); the
  // key is computed only for such points
  T fb[BR_QW];
#pragma unroll
  for (uint32_t t = 0; t < BR_QW; t++) {
    col[t].init(br_lds + Collector::bytes(a.k1) * t, a.k1);
    qid[t] = t < qw ? (a.queries ? a.queries[q0 + t] : q0 + t) : 0u;
#pragma unroll
    for (int j = 0; j < D; j++) qc[t][j] = t < qw ? x[(size_t)j * a.n + qid[t]] : (T)0;
    fb[t] = (T)__builtin_inf();
    if (a.bound && t < qw) {
      col[t].limit(a.bound[q0 + t]);
      fb[t] = (T)(col[t].tk * (1.0 + 0x1p-16) + 0x1p-140);
    }
  }
  const uint64_t c0 = (uint64_t)chunk * a.chunk;
  const uint32_t p0 = (uint32_t)c0;
  const uint32_t p1 = c0 + a.chunk < a.n ? (uint32_t)(c0 + a.chunk) : a.n;
  for (uint32_t base = p0; base < p1; base += 64 * U) {
    T c[U][D];
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
      const uint32_t p = base + 64 * u + lane, pc = p < p1 ? p : p1 - 1u;
#pragma unroll
      for (int j = 0; j < D; j++) c[u][j] = x[(size_t)j * a.n + pc];
    }
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
      const uint32_t p = base + 64 * u + lane;
      const bool valid = p < p1;
#pragma unroll
      for (uint32_t t = 0; t < BR_QW; t++) {
        if (t >= qw) continue;
        if (std::is_same<T, float>::value) {
          // (& and not &&, whose branch per query costs a whole join of 300k 2-D points, K=8, 30.8 ms
          // against 27.3)
          const bool near = valid & (br_dist_sq<D, T>(c[u], qc[t]) <= fb[t]);
          if (__builtin_amdgcn_ballot_w64(near) == 0) continue;
          col[t].offer(near, br_key<D, T>(c[u], qc[t]), p, lane);
          fb[t] = (T)(col[t].tk * (1.0 + 0x1p-16) + 0x1p-140);  // +inf until k1 entries are held
        } else {
          col[t].offer(valid, br_key<D, T>(c[u], qc[t]), p, lane);
        }
      }
    }
  }
#pragma unroll
  for (uint32_t t = 0; t < BR_QW; t++) {
    if (t >= qw) continue;
    col[t].merge(lane);
    if (a.nchunks == 1) {
      br_write_row<T, D>(a, col[t], qid[t], lane);
    } else {
      if (!col[t].nb) continue;
      uint32_t at = 0;
      if (lane == 0) at = atomicAdd(&a.partCount[q0 + t], col[t].nb);
      // (at most k1 entries per chunk: the list has room for all)
      const size_t off = (size_t)(q0 + t) * a.nchunks * a.k1 + (uint32_t)__shfl((int)at, 0, 64);
      for (uint32_t e = lane; e < col[t].nb; e += 64) {
        a.partKey[off + e] = col[t].best_key(e);
        a.partId[off + e] = col[t].best_id(e);
      }
    }
  }
}

template <typename T, int D>
__global__ __launch_bounds__(64) void k_brute_merge(BruteArgs a) {
  extern __shared__ __align__(16) unsigned char br_lds[];
  const uint32_t lane = threadIdx.x;
  const uint32_t qi = blockIdx.x;
  if (qi >= a.nq) return;
  const uint32_t q = a.queries ? a.queries[qi] : qi;
  Collector col;
  col.init(br_lds, a.k1);
  if (a.bound) col.limit(a.bound[qi]);
  const size_t base = (size_t)qi * a.nchunks * a.k1;
  const uint32_t total = a.partCount[qi];
  for (uint32_t e0 = 0; e0 < total; e0 += 256) {
    double k[4];
    uint32_t id[4];
#pragma unroll
    for (uint32_t u = 0; u < 4; u++) {
      const uint32_t e = e0 + 64 * u + lane, ec = e < total ? e : total - 1u;
      k[u] = a.partKey[base + ec];
      id[u] = a.partId[base + ec];
    }
#pragma unroll
    for (uint32_t u = 0; u < 4; u++) col.offer(e0 + 64 * u + lane < total, k[u], id[u], lane);
  }
  col.merge(lane);
  br_write_row<T, D>(a, col, q, lane);
}

size_t br_lds_bytes(uint32_t k1, uint32_t qw) {
  return ((size_t)k1 * 2 * 12 + (size_t)BR_BUF * 12) * qw;
}

template <typename T, int D>
void launch_brute(const BruteArgs &a, hipStream_t s) {
  const uint32_t tiles = (a.nq + a.qw - 1) / a.qw;
  const uint64_t blocks = (uint64_t)tiles * a.nchunks;
  if (a.nchunks > 1) fill_u32(a.partCount, 0u, a.nq, s);
  if (a.bound) k_brute_sample<T, D><<<a.nq, 1024, 0, s>>>(a);
  constexpr uint32_t U = D <= 4 ? 4 : (D <= 8 ? 2 : 1);
  auto partial = a.bound ? k_brute_partial<T, D, U> : k_brute_partial<T, D, 1>;
  partial<<<(uint32_t)blocks, 64, br_lds_bytes(a.k1, a.qw), s>>>(a);
  if (a.nchunks > 1) k_brute_merge<T, D><<<a.nq, 64, br_lds_bytes(a.k1, 1), s>>>(a);
}

__global__ void k_sel_flags(const uint8_t *sel, uint32_t n, uint32_t *flags) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) flags[i] = sel[i] != 0 ? 1u : 0u;
}

__global__ void k_sel_compact(const uint32_t *flags, const uint32_t *pos, uint32_t n, uint32_t *list) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && flags[i]) list[pos[i]] = i;
}

}  // namespace

void select_list(const uint8_t *sel, uint32_t n, uint32_t *flags, uint32_t *pos, uint32_t *list,
                 uint32_t *scratch, hipStream_t s) {
  if (n == 0) return;
  const uint32_t g = (n + 255) / 256;
  k_sel_flags<<<g, 256, 0, s>>>(sel, n, flags);
  scan_exclusive_u32(flags, pos, n, scratch, s);
  k_sel_compact<<<g, 256, 0, s>>>(flags, pos, n, list);
}

BrutePlan brute_plan(uint32_t n, uint32_t nq, uint32_t k1, uint64_t maxPartialEntries) {
  BrutePlan p{};
  if (k1 == 0 || k1 > BRUTE_MAX_K1 || n == 0) return p;
  // queries per wave: as many as the 64 KB LDS budget allows, up to 4
  uint32_t qw = BR_QW;
  while (qw > 1 && br_lds_bytes(k1, qw) > 65536) qw--;
  p.qw = qw;
  const uint32_t tiles = (nq + qw - 1) / qw;
  // enough waves to fill 256 CUs several times over, chunks of at least 16 (K+1) points so
  // the partial lists stay a small fraction of the points scanned
  const uint64_t wantBlocks = 8192;
  uint64_t nchunks = tiles >= wantBlocks ? 1 : (wantBlocks + tiles - 1) / tiles;
  uint64_t minChunk = (uint64_t)k1 * 16 > 1024 ? (uint64_t)k1 * 16 : 1024;
  uint64_t maxChunks = (n + minChunk - 1) / minChunk;
  if (nchunks > maxChunks) nchunks = maxChunks;
  if (nchunks == 0) nchunks = 1;
  // partial tables within maxPartialEntries entries (12 bytes each)
  const uint64_t memChunks = (maxPartialEntries / ((uint64_t)nq * k1)) > 0 ? (maxPartialEntries / ((uint64_t)nq * k1)) : 1;
  if (nchunks > memChunks) nchunks = memChunks;
  uint64_t chunk = (n + nchunks - 1) / nchunks;
  chunk = (chunk + 63) & ~63ull;
  nchunks = (n + chunk - 1) / chunk;
  if (tiles * nchunks > 0x7fffffffull) return BrutePlan{};
  p.chunk = (uint32_t)chunk;
  p.nchunks = (uint32_t)nchunks;
  p.partialEntries = nchunks > 1 ? (uint64_t)nq * nchunks * k1 : 0;
  // sample: a round of 64 points then holds one within the bound (its FP64 key and the collector
  // cost several times the filter) in about an eighth of the rounds, and at most 8192 points in all
  // do.  Past 4096 queries the chunks are few and long, and the samples cost as much as they save
  // (763 queries over 1M 6-D points, K=32: scan without a bound 1.43 ms, with it 0.68 + 0.07).
  const uint64_t m = std::max<uint64_t>({(uint64_t)n * k1 / 8192, 512ull * k1, 1024}) & ~63ull;
  p.sample = nchunks > 1 && nq <= BR_SAMPLE_NQ && m >= k1 && m <= n / 4 ? (uint32_t)m : 0u;
  return p;
}

template <typename T>
void brute_join(const BruteArgs &a, hipStream_t s) {
  if (a.nq == 0) return;
  switch (a.d) {
    case 1: launch_brute<T, 1>(a, s); break;
    case 2: launch_brute<T, 2>(a, s); break;
    case 3: launch_brute<T, 3>(a, s); break;
    case 4: launch_brute<T, 4>(a, s); break;
    case 5: launch_brute<T, 5>(a, s); break;
    case 6: launch_brute<T, 6>(a, s); break;
    case 7: launch_brute<T, 7>(a, s); break;
    case 8: launch_brute<T, 8>(a, s); break;
    case 9: launch_brute<T, 9>(a, s); break;
    case 10: launch_brute<T, 10>(a, s); break;
    case 11: launch_brute<T, 11>(a, s); break;
    case 12: launch_brute<T, 12>(a, s); break;
    case 13: launch_brute<T, 13>(a, s); break;
    case 14: launch_brute<T, 14>(a, s); break;
    case 15: launch_brute<T, 15>(a, s); break;
    case 16: launch_brute<T, 16>(a, s); break;
    default: break;
  }
}

template void brute_join<float>(const BruteArgs &, hipStream_t);
template void brute_join<double>(const BruteArgs &, hipStream_t);

}  // namespace knn
