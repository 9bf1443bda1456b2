// batched.hip -- many independent point sets joined together (float32).
//
// No counterpart in the reference, which joins one set per process (main.cu:109-510).  The
// sets of one dimensionality and range kernel form a group; the group's points are concatenated
// and every stage runs once per group over all of them:
//   per-set variance reorder (main.cu:2521-2615, same FP32 sums as a single-set join),
//   per-set min/max, per-set grid (own width, own key range [keyBase, keyBase + cells)),
//   one radix sort / cell table / dense start table for the whole group,
//   tiles of queries of one set, and the range kernels with per-tile set descriptors (grid,
//   K+1, row offset).
// Radius schedule (per query, any schedule gives the same rows): each set first gets a grid of
// width wf (about K+1 points per cell at its mean density); a query's initial radius is the
// one whose ball holds about 2 (K+1) points at the density of its own and the two adjacent
// cells along dim 0.  Then passes over radius classes: in each pass every set joins its
// pending queries of its lowest occupied class (class_bins quarter octaves) on a grid matched to
// the class's largest radius; failed queries grow their radius.
// Rows are exact whatever the radii (a query is accepted only when its K+1 nearest are
// provably inside its block) and equal the rows of a single-set join of the same set.
//
// Every kernel reads its sizes (cells, tiles) from device memory, so a pass is a fixed
// sequence of launches: a group's set-up and first pass, a further pass, and the overflow kernel's
// part are captured once in hipGraphs and replayed for later calls with the same set shapes, on a
// stream per group, each pass only while queries of the group are pending.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "knn_launch.h"

namespace knn {

namespace {

constexpr uint32_t BLK = 256;
inline uint32_t nblk(size_t n) { return (uint32_t)((n + BLK - 1) / BLK); }

// main.cu:2537-2562 per set: rows 0,100,... of the set summed in order per dim.  One wave per set:
// 64 sampled rows at a time go to LDS (lane = row, the next 64 in flight), then lane = dim adds
// them in order: 50 us per group of 12 sets of up to 200k points.  (A thread per (set, dim) that
// reads each row as it comes waits out a memory round trip per addition: 595 us.)
__global__ __launch_bounds__(64) void k_b_variance(const float *__restrict__ xin, const SetDesc *sets,
                                                   uint32_t d, float *var) {
  __shared__ float rows[64 * (KNN_MAXDIM + 1)];
  const uint32_t si = blockIdx.x, lane = threadIdx.x;
  const uint32_t n = sets[si].n;
  const float *pts = xin + (size_t)sets[si].pStart * d;
  const float inv = (float)(1.0 / (100 * 1.0));
  const float denom = (float)n * inv;
  const uint32_t m = (uint32_t)(((uint64_t)n + 99) / 100);  // sampled rows
  float avg = 0.0f;
  for (int pass = 0; pass < 2; pass++) {
    float sum = 0.0f;
    float nx[KNN_MAXDIM];
    auto load = [&](uint32_t r0) {
      const uint32_t r = r0 + lane < m ? r0 + lane : m - 1u;
#pragma unroll
      for (uint32_t k = 0; k < KNN_MAXDIM; k++)
        if (k < d) nx[k] = pts[(uint64_t)r * 100u * d + k];
    };
    if (m) load(0);
    for (uint32_t r0 = 0; r0 < m; r0 += 64) {
      __syncthreads();  // the previous rows have been added
#pragma unroll
      for (uint32_t k = 0; k < KNN_MAXDIM; k++)
        if (k < d) rows[lane * (KNN_MAXDIM + 1) + k] = nx[k];
      __syncthreads();
      if (r0 + 64 < m) load(r0 + 64);
      const uint32_t c = m - r0 < 64u ? m - r0 : 64u;
      if (lane < d) {
#pragma unroll 16
        for (uint32_t r = 0; r < c; r++) {
          const float x = rows[r * (KNN_MAXDIM + 1) + lane];
          if (pass == 0) {
            sum += x;
          } else {
            const float df = x - avg;
            const float sq = df * df;
            sum += sq;
          }
        }
      }
    }
    if (pass == 0) avg = sum / denom;
    else if (lane < d) var[(size_t)si * d + lane] = sum / denom;
  }
}

// stable descending insertion sort of each set's variances (main.cu:2580)
__global__ void k_b_perm(const float *var, uint32_t nsets, uint32_t d, int reorder, uint32_t *perm) {
  const uint32_t si = blockIdx.x * blockDim.x + threadIdx.x;
  if (si >= nsets) return;
  uint32_t p[KNN_MAXDIM];
  for (uint32_t i = 0; i < d; i++) p[i] = i;
  if (reorder) {
    const float *v = var + (size_t)si * d;
    for (uint32_t i = 1; i < d; i++) {
      const uint32_t pi = p[i];
      const float key = v[pi];
      int j = (int)i - 1;
      while (j >= 0 && key > v[p[j]]) {
        p[j + 1] = p[j];
        j--;
      }
      p[j + 1] = pi;
    }
  }
  for (uint32_t i = 0; i < KNN_MAXDIM; i++) perm[(size_t)si * KNN_MAXDIM + i] = i < d ? p[i] : 0u;
}

__global__ void k_b_permute(const float *__restrict__ xin, uint32_t N, uint32_t d,
                            const uint32_t *__restrict__ setOf, const uint32_t *__restrict__ perm,
                            float *__restrict__ x) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= N) return;
  const uint32_t *pm = perm + (size_t)setOf[p] * KNN_MAXDIM;
  for (uint32_t j = 0; j < d; j++) x[(size_t)j * N + p] = xin[(size_t)p * d + pm[j]];
}

// one block per (set, indexed dim): min / max -> mnmx[si][0..7] min, [8..15] max.  14 us per group
// of 12 sets of up to 200k points (256 threads per set, one dim after the other: 454 us)
__global__ __launch_bounds__(1024) void k_b_minmax(const float *__restrict__ x, uint32_t N,
                                                   const SetDesc *sets, float *mnmx) {
  __shared__ float smn[16], smx[16];
  const SetDesc &sd = sets[blockIdx.x];
  const uint32_t j = blockIdx.y;
  if (j >= sd.nd) return;
  const float *col = x + (size_t)j * N + sd.pStart;
  float mn = __builtin_inff(), mx = -__builtin_inff();
#pragma unroll 4
  for (uint32_t i = threadIdx.x; i < sd.n; i += 1024) {
    const float v = col[i];
    mn = fminf(mn, v);
    mx = fmaxf(mx, v);
  }
  for (int o = 32; o > 0; o >>= 1) {
    mn = fminf(mn, __shfl_xor(mn, o, 64));
    mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  }
  if ((threadIdx.x & 63) == 0) {
    smn[threadIdx.x >> 6] = mn;
    smx[threadIdx.x >> 6] = mx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 16; w++) {
      mn = fminf(mn, smn[w]);
      mx = fmaxf(mx, smx[w]);
    }
    mnmx[(size_t)blockIdx.x * 16 + j] = mn;
    mnmx[(size_t)blockIdx.x * 16 + 8 + j] = mx;
  }
}

__device__ double unit_ball_volume(uint32_t nd) {
  // V_1 = 2, V_2 = pi, V_n = V_{n-2} * 2 pi / n
  double v = (nd & 1) ? 2.0 : 3.14159265358979323846;
  for (uint32_t m = (nd & 1) ? 3 : 4; m <= nd; m += 2) v *= 2.0 * 3.14159265358979323846 / m;
  return v;
}

// Per set: wf = (V (K+1) / n)^(1/nd) over its bounding box (degenerate boxes: largest extent / 8,
// or 1); the first grid uses it.  All queries pending.
__global__ void k_b_init_width(SetDesc *sets, uint32_t nsets, const float *mnmx, float *width,
                               uint32_t *setMinBin) {
  const uint32_t si = blockIdx.x * blockDim.x + threadIdx.x;
  if (si >= nsets) return;
  SetDesc &sd = sets[si];
  double vol = 1.0, ext = 0.0;
  for (uint32_t j = 0; j < sd.nd; j++) {
    const double e = (double)mnmx[(size_t)si * 16 + 8 + j] - (double)mnmx[(size_t)si * 16 + j];
    vol *= e;
    ext = e > ext ? e : ext;
  }
  double w = 0.0;
  if (vol > 0.0 && sd.n > 0) w = pow((double)sd.k1 * vol / (double)sd.n, 1.0 / sd.nd);
  if (!(w > 0.0) || !(w < 3.0e38)) w = ext > 0.0 ? ext / 8.0 : 1.0;
  float wf = (float)w;
  if (!(wf > 0.0f)) wf = 1.0f;
  sd.r0 = wf;
  width[si] = wf;
  setMinBin[si] = 64u;
}

__global__ void k_b_pending(uint32_t N, uint8_t *failed) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < N) failed[p] = 1;
}

// quarter-octave bin of r relative to wf: floor(4 log2(r / wf)) + 32 in [0, 63]
__device__ __forceinline__ int bin_of(float r, float wf) {
  const float x = 4.0f * log2f(r / wf);
  if (!(x >= -32.0f)) return 0;
  if (x >= 31.0f) return 63;
  const int b = (int)floorf(x) + 32;
  return b < 0 ? 0 : (b > 63 ? 63 : b);
}

// Lowest bin of the pending queries of each set, from a block of 256 threads that holds
// consecutive points: one atomic per block where all its points are of one set (lo == hi, the
// sets of its first and last point), else one per wave and set present.  key = set << 8 | bin
// (~0: not pending).  The minimum only falls, so a reader of one already as low needs no atomic.
// (A pass over the points of its own with an atomic per wave, all on a few words, took 55 us per
// pass of 12 sets of up to 200k points; as part of k_b_grow_class it and the counting take 7 us.)
__device__ __forceinline__ void lower_min_bin(uint32_t *setMinBin, uint32_t si, uint32_t b) {
  if (b < __hip_atomic_load(&setMinBin[si], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    atomicMin(&setMinBin[si], b);
}
__device__ __forceinline__ void block_min_bin(uint32_t key, uint32_t lo, uint32_t hi, uint32_t *setMinBin,
                                              uint32_t *lds4) {
  if (lo == hi) {  // block-uniform
    uint32_t b = key;
    for (int o = 32; o > 0; o >>= 1) {
      const uint32_t t = (uint32_t)__shfl_xor((int)b, o, 64);
      b = t < b ? t : b;
    }
    if ((threadIdx.x & 63) == 0) lds4[threadIdx.x >> 6] = b;
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int w = 1; w < 4; w++) b = lds4[w] < b ? lds4[w] : b;
      if (b != 0xffffffffu) lower_min_bin(setMinBin, lo, b & 0xffu);
    }
    return;
  }
  bool mine = key != 0xffffffffu;
  for (;;) {
    const uint64_t live = __ballot(mine);
    if (!live) break;
    const int leader = __ffsll((long long)live) - 1;
    const uint32_t ls = (uint32_t)__shfl((int)(key >> 8), leader, 64);
    uint32_t b = (mine && (key >> 8) == ls) ? (key & 0xffu) : 0xffu;
    for (int o = 32; o > 0; o >>= 1) {
      const uint32_t t = (uint32_t)__shfl_xor((int)b, o, 64);
      b = t < b ? t : b;
    }
    if ((int)(threadIdx.x & 63) == leader) lower_min_bin(setMinBin, ls, b);
    if ((key >> 8) == ls) mine = false;
  }
}

// Initial radius of every query from the points of its own and the two adjacent cells along
// dim 0 on the wf grid: density rho = count / volume, r = (2 (K+1) / (V_nd rho))^(1/nd),
// kept within [wf / 64, 64 wf].
__global__ __launch_bounds__(256) void k_b_density_radius(const float *__restrict__ x, uint32_t N,
                                                          const SetDesc *sets, const uint32_t *__restrict__ setOf,
                                                          const uint32_t *__restrict__ dense, float *radius,
                                                          uint8_t *bin, uint32_t *setMinBin) {
  __shared__ uint32_t lds4[4];
  const uint32_t first = blockIdx.x * 256u, q = first + threadIdx.x;
  const uint32_t lo = setOf[first], hi = setOf[first + 255u < N ? first + 255u : N - 1u];
  uint32_t key = 0xffffffffu;
  if (q < N) {
    const uint32_t si = setOf[q];
    const SetDesc &sd = sets[si];
    const GridParams &g = sd.g;
    uint64_t row = g.keyBase;
    uint32_t c0 = 0;
    for (uint32_t j = 0; j < g.nd; j++) {
      const uint32_t c = cell_coord<float>(x[(size_t)j * N + q], g.minArr[j], g.eps, g.nCells[j]);
      if (j == 0) c0 = c; else row += (uint64_t)c * g.mult[j];
    }
    const uint32_t cl = c0 > 0 ? c0 - 1 : 0;
    const uint32_t ch = c0 + 1 < g.nCells[0] ? c0 + 1 : g.nCells[0] - 1;
    const uint32_t cnt = dense[row + ch + 1] - dense[row + cl];
    const double wf = (double)sd.r0;
    const double vol = (double)(ch - cl + 1) * pow((double)g.eps, (double)g.nd);
    const double rho = (double)(cnt > 0 ? cnt : 1u) / vol;
    double r = pow(2.0 * sd.k1 / (unit_ball_volume(g.nd) * rho), 1.0 / g.nd);
    r = fmin(fmax(r, wf / 64.0), wf * 64.0);
    const int b = bin_of((float)r, sd.r0);
    radius[q] = (float)r;
    bin[q] = (uint8_t)b;
    key = (si << 8) | (uint32_t)b;
  }
  block_min_bin(key, lo, hi, setMinBin, lds4);
}

// Radius classes: quarter-octave bins per class and cells per class radius R, by the number of
// indexed dims.  A class costs an index build over all N points of the group, a wide one larger
// blocks for its small radii (what lies outside a query's ball is cut by cells, so fine cells
// cost little).  48 sets of 1k-200k points, 30 % of them in tight clusters, ms of each group
// alone with bins / div of 10 / 4, 12 / 5 and 16 / 6 in 2-D: 3.74, 3.62, 3.01; 5 / 1.5, 8 / 2 and
// 10 / 2.5 in 4-D: 4.7, 4.56, 4.38; 4 / 1.5, 6 / 2 and 5 / 1.5 in 6-D (second mix): 8.60, 8.12, 7.70.
__host__ __device__ __forceinline__ uint32_t class_bins(uint32_t nd) { return nd <= 2 ? 16u : (nd <= 4 ? 10u : 5u); }
__device__ __forceinline__ double class_div(uint32_t nd) { return nd <= 2 ? 6.0 : (nd <= 4 ? 2.5 : 1.5); }

// aflags[p] = the point at sorted position p is pending with a radius in its set's class
__global__ void k_b_class_flags(const uint32_t *__restrict__ sortedIds, const uint32_t *__restrict__ setOf,
                                const uint8_t *__restrict__ failed, const uint8_t *__restrict__ bin,
                                const uint32_t *__restrict__ setClass, uint32_t bins, uint32_t N,
                                uint32_t *__restrict__ aflags) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= N) return;
  const uint32_t q = sortedIds[p];
  const uint32_t c = setClass[setOf[q]], b = bin[q];
  aflags[p] = failed[q] && b >= c && b < c + bins ? 1u : 0u;
}

// End of a pass: its failed queries (of the class; OVER: those the overflow kernel took, which
// the class's own step leaves alone) grow their radius, an octave or half an octave with >= 3
// indexed dims; queries still pending into *pending, their lowest bins into setMinBin.  Blocks
// of 1024 consecutive points.
constexpr uint32_t GROW_PTS = 1024;
template <bool OVER>
__global__ __launch_bounds__(256) void k_b_grow_class(const SetDesc *sets, const uint32_t *__restrict__ setOf,
                                                      const uint32_t *__restrict__ setClass, uint32_t bins,
                                                      const uint8_t *__restrict__ failed, uint8_t *overflow,
                                                      uint32_t N, float *radius, uint8_t *bin, uint32_t *pending,
                                                      uint32_t *setMinBin) {
  __shared__ uint32_t lds4[4], sum[4];
  const uint32_t first = blockIdx.x * GROW_PTS;
  const uint32_t last = N - first < GROW_PTS ? N - 1u : first + GROW_PTS - 1u;
  const uint32_t lo = setOf[first], hi = setOf[last];
  uint32_t cnt = 0, low = 0xffffffffu;
  for (uint32_t u = 0; u < GROW_PTS / 256; u++) {
    const uint32_t q = first + u * 256u + threadIdx.x;
    uint32_t key = 0xffffffffu;
    if (q <= last) {
      const bool ov = overflow[q];
      if (failed[q]) {
        const uint32_t si = setOf[q], c = setClass[si];
        uint32_t b = bin[q];
        cnt++;
        if (OVER ? ov : (!ov && b >= c && b < c + bins)) {
          const float r = radius[q] * (sets[si].nd <= 2 ? 2.0f : 1.41421356f);
          radius[q] = r;
          // at least one bin further, so that every failure moves the query to a later class
          const uint32_t nb = (uint32_t)bin_of(r, sets[si].r0);
          b = nb > b ? nb : (b + 1u < 64u ? b + 1u : 63u);
          bin[q] = (uint8_t)b;
        }
        key = (si << 8) | b;
      }
      if (OVER && ov) overflow[q] = 0;
    }
    if (lo == hi) low = key < low ? key : low;
    else block_min_bin(key, lo, hi, setMinBin, lds4);
  }
  if (lo == hi) block_min_bin(low, lo, hi, setMinBin, lds4);
  for (int o = 32; o > 0; o >>= 1) cnt += (uint32_t)__shfl_xor((int)cnt, o, 64);
  if ((threadIdx.x & 63) == 0) sum[threadIdx.x >> 6] = cnt;
  __syncthreads();
  if (threadIdx.x == 0) {
    cnt = sum[0] + sum[1] + sum[2] + sum[3];
    if (cnt) atomicAdd(pending, cnt);
  }
}

// One wave, lane = set (64 at a time).  With setMinBin, first every set's radius class, the
// lowest bin c of its pending queries and the class_bins - 1 above, and its width R / class_div
// (R = the class's upper radius; sets without pending queries keep their width); setMinBin is
// cleared for the pass's own failures.  Then the grid of every set at its width
// (main.cu:2465-2486 arithmetic: lo = min - w, nCells = ceil((max + w - lo) / w)); the key ranges
// are laid end to end.  When the total would exceed `bound` cells, every width grows by 1/4 until
// it fits.  5 us at 12 sets (14 us with one thread taking them in turn).
__global__ __launch_bounds__(64) void k_b_grids(SetDesc *sets, uint32_t nsets, const float *mnmx, float *width,
                                                uint64_t bound, uint32_t *status, uint32_t *setMinBin,
                                                uint32_t *setClass) {
  const uint32_t lane = threadIdx.x;
  if (setMinBin)
    for (uint32_t si = lane; si < nsets; si += 64) {
      const uint32_t c = setMinBin[si];
      setClass[si] = c;
      setMinBin[si] = 64u;
      if (c >= 64) continue;
      const double R = (double)sets[si].r0 * exp2(((double)c + class_bins(sets[si].nd) - 32.0) / 4.0);
      width[si] = (float)(R / class_div(sets[si].nd));
    }
  for (int attempt = 0; attempt < 256; attempt++) {
    uint64_t base = 0;
    bool fits = true;
    for (uint32_t s0 = 0; s0 < nsets && fits; s0 += 64) {
      const uint32_t si = s0 + lane;
      uint64_t tot = 0;
      if (si < nsets) {
        SetDesc &sd = sets[si];
        const float w = width[si];
        GridParams &g = sd.g;
        g.eps = w;
        g.nd = sd.nd;
        tot = 1;
        for (uint32_t j = 0; j < KNN_MAX_INDEXED; j++) {
          if (j < sd.nd) {
            const float lo = mnmx[(size_t)si * 16 + j] - w;
            const float hi = mnmx[(size_t)si * 16 + 8 + j] + w;
            const float q = (hi - lo) / w;
            float c = ceilf(q);
            if (!(c >= 1.0f)) c = 1.0f;
            if (c > 2147483647.0f) c = 2147483647.0f;
            g.minArr[j] = lo;
            g.nCells[j] = (uint32_t)c;
            g.mult[j] = tot;
            tot *= (uint64_t)g.nCells[j];
            if (tot > bound) break;
          } else {
            g.minArr[j] = 0.0f;
            g.nCells[j] = 1;
            g.mult[j] = tot;
          }
        }
      }
      // a total past bound stops the attempt, so the sums stay far below 2^64
      fits = !__any(tot > bound);
      if (fits) {
        uint64_t incl = tot;
        for (int o = 1; o < 64; o <<= 1) {
          const uint64_t t = __shfl_up(incl, o, 64);
          if ((int)lane >= o) incl += t;
        }
        if (si < nsets) sets[si].g.keyBase = base + incl - tot;
        base += __shfl(incl, 63, 64);
        fits = base <= bound;
      }
    }
    if (fits) {
      if (lane == 0) {
        status[0] = 0;
        status[1] = (uint32_t)base;
      }
      return;
    }
    for (uint32_t si = lane; si < nsets; si += 64) width[si] *= 1.25f;
  }
  // no fit (only with very many sets of many indexed dims): one cell per set, keys 0..nsets-1
  // (bound >= 8 N >= nsets); every query then scans its whole set, which is slow but exact
  for (uint32_t si = lane; si < nsets; si += 64) {
    GridParams &g = sets[si].g;
    g.keyBase = si;
    g.nd = sets[si].nd;
    for (uint32_t j = 0; j < KNN_MAX_INDEXED; j++) {
      g.minArr[j] = 0.0f;
      g.nCells[j] = 1;
      g.mult[j] = 1;
    }
  }
  if (lane == 0) {
    status[0] = 1;
    status[1] = nsets;
  }
}

__global__ void k_b_cell_keys(const float *__restrict__ x, uint32_t N, const SetDesc *sets,
                              const uint32_t *__restrict__ setOf, uint32_t *keys, uint32_t *ids) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= N) return;
  const GridParams &g = sets[setOf[p]].g;
  uint64_t id = g.keyBase;
  for (uint32_t j = 0; j < g.nd; j++)
    id += (uint64_t)cell_coord<float>(x[(size_t)j * N + p], g.minArr[j], g.eps, g.nCells[j]) * g.mult[j];
  keys[p] = (uint32_t)id;
  ids[p] = p;
}

// dense[cellKeys[c]] = points of cell c, for c < *ncell
__global__ void k_b_dense_counts(const uint64_t *cellKeys, const uint32_t *cellStart,
                                 const uint32_t *ncell, uint32_t N, uint32_t *dense) {
  const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= N || c >= *ncell) return;
  dense[cellKeys[c]] = cellStart[c + 1] - cellStart[c];
}

__global__ void k_b_flags_u8(const uint32_t *sortedIds, const uint8_t *f, uint32_t N, uint32_t *flags) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= N) return;
  flags[p] = f[sortedIds[p]] ? 1u : 0u;
}

// tiles of <= tq active queries per non-empty cell (cells c < *ncell; entries up to N + 1)
__global__ void k_b_tile_counts(const uint32_t *cellStart, const uint32_t *pos, const uint32_t *ncell,
                                uint32_t N, uint32_t tq, uint32_t *ntiles) {
  const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c > N) return;
  if (c >= *ncell) {
    ntiles[c] = 0;
    return;
  }
  const uint32_t a0 = pos[cellStart[c]], a1 = pos[cellStart[c + 1]];
  ntiles[c] = (a1 - a0 + tq - 1) / tq;
}

__global__ void k_b_write_tiles(const uint32_t *cellStart, const uint32_t *pos, const uint32_t *tileOff,
                                const uint32_t *ncell, uint32_t N, uint32_t tq, uint2 *tiles) {
  const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= N || c >= *ncell) return;
  const uint32_t a0 = pos[cellStart[c]], a1 = pos[cellStart[c + 1]];
  uint32_t t = tileOff[c];
  for (uint32_t a = a0; a < a1; a += tq, t++) {
    const uint32_t m = (a1 - a < tq) ? a1 - a : tq;
    tiles[t] = make_uint2(a, m);
  }
}

// Tiles of the direct kernel: chunks of up to q consecutive active queries of one set, whatever
// their cells.  The keys are laid out set after set, so set si holds the sorted positions
// [pStart, pStart + n) and its active queries are act[pos[pStart] .. pos[pStart + n]).  (Tiles
// that end with their cell hold a few queries each on grids this fine, and the kernel looks up the
// rows of 64 at a time: 5.5 ms against 1.8 for a 2-D group of 12 sets of up to 200k points.)  q is
// small enough for each of `waves` waves to take a chunk, at most cap.  One block: chunkOff[si]
// = chunks before set si, *ntiles = all of them, qOut = q.
__global__ __launch_bounds__(256) void k_b_chunk_offsets(const SetDesc *sets, uint32_t nsets,
                                                         const uint32_t *__restrict__ pos, uint32_t N,
                                                         uint32_t waves, uint32_t cap, uint32_t *chunkOff,
                                                         uint32_t *ntiles, uint32_t *qOut) {
  __shared__ uint32_t part[4];
  const uint32_t A = pos[N], lane = threadIdx.x & 63;
  uint32_t q = A / waves;
  q = q < 1u ? 1u : (q > cap ? cap : q);
  uint32_t base = 0;
  for (uint32_t s0 = 0; s0 < nsets; s0 += 256) {
    const uint32_t si = s0 + threadIdx.x;
    uint32_t c = 0;
    if (si < nsets) c = (pos[sets[si].pStart + sets[si].n] - pos[sets[si].pStart] + q - 1u) / q;
    uint32_t incl = c;
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t t = (uint32_t)__shfl_up((int)incl, o, 64);
      if ((int)lane >= o) incl += t;
    }
    __syncthreads();
    if (lane == 63) part[threadIdx.x >> 6] = incl;
    __syncthreads();
    uint32_t before = base;
    for (uint32_t w = 0; w < 4; w++) {
      if (w < threadIdx.x >> 6) before += part[w];
      base += part[w];
    }
    if (si < nsets) chunkOff[si] = before + incl - c;
  }
  if (threadIdx.x == 0) {
    chunkOff[nsets] = base;
    *ntiles = base;
    *qOut = q;
  }
}

// tiles[t] = chunk t: thread per chunk, its set by binary search (at most N chunks: every chunk
// holds a query)
__global__ void k_b_chunks(const SetDesc *sets, uint32_t nsets, const uint32_t *__restrict__ pos,
                           const uint32_t *__restrict__ chunkOff, const uint32_t *qIn, uint2 *tiles) {
  const uint32_t q = *qIn, n = chunkOff[nsets];
  for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
    uint32_t l = 0, h = nsets;  // chunkOff[l] <= t < chunkOff[h]
    while (h - l > 1) {
      const uint32_t m = (l + h) / 2;
      if (chunkOff[m] <= t) l = m; else h = m;
    }
    const uint32_t a0 = pos[sets[l].pStart] + (t - chunkOff[l]) * q, a1 = pos[sets[l].pStart + sets[l].n];
    const uint32_t m = a1 - a0 < q ? a1 - a0 : q;
    tiles[t] = make_uint2(a0, m);
  }
}

}  // namespace

// ------------------------------------------------------------------ host launchers
void batch_variance_perm(const float *xin, const SetDesc *sets, uint32_t nsets, uint32_t d, int reorder,
                         float *var, uint32_t *perm, hipStream_t s) {
  if (nsets) k_b_variance<<<nsets, 64, 0, s>>>(xin, sets, d, var);
  k_b_perm<<<nblk(nsets), BLK, 0, s>>>(var, nsets, d, reorder, perm);
}
void batch_permute(const float *xin, uint32_t N, uint32_t d, const uint32_t *setOf, const uint32_t *perm,
                   float *x, hipStream_t s) {
  if (N) k_b_permute<<<nblk(N), BLK, 0, s>>>(xin, N, d, setOf, perm, x);
}
void batch_minmax(const float *x, uint32_t N, const SetDesc *sets, uint32_t nsets, float *mnmx,
                  hipStream_t s) {
  if (nsets) k_b_minmax<<<dim3(nsets, KNN_MAX_INDEXED), 1024, 0, s>>>(x, N, sets, mnmx);
}
void batch_init_width(SetDesc *sets, uint32_t nsets, const float *mnmx, float *width, uint32_t *setMinBin,
                      uint32_t N, uint8_t *failed, hipStream_t s) {
  k_b_init_width<<<nblk(nsets), BLK, 0, s>>>(sets, nsets, mnmx, width, setMinBin);
  if (N) k_b_pending<<<nblk(N), BLK, 0, s>>>(N, failed);
}
void batch_density_radius(const float *x, uint32_t N, const SetDesc *sets, const uint32_t *setOf,
                          const uint32_t *dense, float *radius, uint8_t *bin, uint32_t *setMinBin, hipStream_t s) {
  if (N) k_b_density_radius<<<nblk(N), BLK, 0, s>>>(x, N, sets, setOf, dense, radius, bin, setMinBin);
}
void batch_class_flags(const uint32_t *sortedIds, const uint32_t *setOf, const uint8_t *failed, const uint8_t *bin,
                       const uint32_t *setClass, uint32_t nd, uint32_t N, uint32_t *aflags, hipStream_t s) {
  if (N) k_b_class_flags<<<nblk(N), BLK, 0, s>>>(sortedIds, setOf, failed, bin, setClass, class_bins(nd), N, aflags);
}
void batch_grow_class(const SetDesc *sets, const uint32_t *setOf, const uint32_t *setClass, uint32_t nd,
                      const uint8_t *failed, uint8_t *overflow, bool over, uint32_t N, float *radius, uint8_t *bin,
                      uint32_t *pending, uint32_t *setMinBin, hipStream_t s) {
  if (!N) return;
  const uint32_t nb = (N + GROW_PTS - 1) / GROW_PTS;
  auto kern = over ? k_b_grow_class<true> : k_b_grow_class<false>;
  kern<<<nb, 256, 0, s>>>(sets, setOf, setClass, class_bins(nd), failed, overflow, N, radius, bin, pending, setMinBin);
}
void batch_grids(SetDesc *sets, uint32_t nsets, const float *mnmx, float *width, uint64_t bound,
                 uint32_t *status, uint32_t *setMinBin, uint32_t *setClass, hipStream_t s) {
  k_b_grids<<<1, 64, 0, s>>>(sets, nsets, mnmx, width, bound, status, setMinBin, setClass);
}
void batch_cell_keys(const float *x, uint32_t N, const SetDesc *sets, const uint32_t *setOf,
                     uint32_t *keys, uint32_t *ids, hipStream_t s) {
  if (N) k_b_cell_keys<<<nblk(N), BLK, 0, s>>>(x, N, sets, setOf, keys, ids);
}
void batch_dense_counts(const uint64_t *cellKeys, const uint32_t *cellStart, const uint32_t *ncell,
                        uint32_t N, uint32_t *dense, hipStream_t s) {
  if (N) k_b_dense_counts<<<nblk(N), BLK, 0, s>>>(cellKeys, cellStart, ncell, N, dense);
}
void batch_flags_u8(const uint32_t *sortedIds, const uint8_t *f, uint32_t N, uint32_t *flags, hipStream_t s) {
  if (N) k_b_flags_u8<<<nblk(N), BLK, 0, s>>>(sortedIds, f, N, flags);
}
void batch_tiles(const uint32_t *cellStart, const uint32_t *pos, const uint32_t *ncell, uint32_t N,
                 uint32_t tq, uint32_t *ntiles, uint32_t *tileOff, uint32_t *scratch, uint2 *tiles,
                 hipStream_t s) {
  k_b_tile_counts<<<nblk((size_t)N + 1), BLK, 0, s>>>(cellStart, pos, ncell, N, tq, ntiles);
  scan_exclusive_u32(ntiles, tileOff, N + 1, scratch, s);
  if (N) k_b_write_tiles<<<nblk(N), BLK, 0, s>>>(cellStart, pos, tileOff, ncell, N, tq, tiles);
}
void batch_chunks(const SetDesc *sets, uint32_t nsets, uint32_t nd, const uint32_t *pos, uint32_t N, uint32_t waves, uint32_t cap,
                  uint32_t *chunkOff, uint32_t *ntiles, uint32_t *q, uint2 *tiles, hipStream_t s) {
  // chunks per wave: a query's time grows with its indexed dims and with it the cost of an uneven
  // end (6-D group of a 48-set mix: 12.2 ms with 1, 9.3 with 4, 8.1 with 8;
  // 2-D chunks look up the rows of 64 queries at a time, so that smaller ones waste lanes)
  const uint32_t per = nd <= 2 ? 1u : (nd <= 4 ? 4u : 8u);
  k_b_chunk_offsets<<<1, 256, 0, s>>>(sets, nsets, pos, N, waves * per, cap, chunkOff, ntiles, q);
  k_b_chunks<<<std::min<uint32_t>(nblk(N), 256u), BLK, 0, s>>>(sets, nsets, pos, chunkOff, q, tiles);
}
}  // namespace knn
