// join.hip -- grid index, active-query tiles and the checksum reduction for gfx950.
//
// Index (replaces GPU.cu:3715-4067): per-point cell key (kernel.cu:1673-1697) -> stable LSD
// radix sort of (key, point id) (prims.hip) -> boundary flags + scan -> compacted non-empty
// cell table {cellKeys[c], cellStart[c]} in HBM, plus a cell-sorted dim-major copy of the
// coordinates (xs) so that every candidate range is one contiguous, coalesced stream.
//
#include "knn_range.h"

namespace knn {

namespace {

// ------------------------------------------------------------------ index kernels
template <typename T, typename K, typename G>
__global__ void k_cell_keys(const T *__restrict__ x, uint32_t n, G g, K *keys, uint32_t *ids) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint64_t id = 0;
  for (uint32_t j = 0; j < g.nd; j++) {
    uint32_t c = cell_coord<T>(x[(size_t)j * n + i], (T)g.minArr[j], (T)g.eps, g.nCells[j]);
    id += (uint64_t)c * g.mult[j];
  }
  // slab order: the cell id above the slab code of the first non-indexed dim (one sort gives
  // cell order, and slab order within each cell)
  if (g.sb) id = (id << g.sb) | slab_q<T>(x[(size_t)g.nd * n + i], g);
  keys[i] = (K)id;
  ids[i] = i;
}

// sb: the slab code's bits below the cell id in the keys (0 without slab order)
template <typename K>
__global__ void k_boundary_flags(const K *keys, uint32_t n, uint32_t sb, uint32_t *flags) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  flags[p] = (p == 0 || (keys[p] >> sb) != (keys[p - 1] >> sb)) ? 1u : 0u;
}

template <typename K>
__global__ void k_compact_cells(const K *keys, const uint32_t *flags, const uint32_t *pos,
                                uint32_t n, uint32_t sb, uint64_t *cellKeys, uint32_t *cellStart) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  if (flags[p]) {
    cellKeys[pos[p]] = (uint64_t)(keys[p] >> sb);
    cellStart[pos[p]] = p;
  }
  if (p == n - 1) cellStart[pos[n]] = n;
}

template <typename T>
__global__ void k_gather_soa(const T *__restrict__ x, const uint32_t *__restrict__ ids, uint32_t n,
                             uint32_t d, T *__restrict__ xs) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const uint32_t i = ids[p];
  for (uint32_t j = 0; j < d; j++) xs[(size_t)j * n + p] = x[(size_t)j * n + i];
}

__global__ void k_gather_u32(const uint32_t *__restrict__ src, const uint32_t *__restrict__ idx, uint32_t n,
                             uint32_t *__restrict__ dst) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n) dst[p] = src[idx[p]];
}

// xs[j*n + p] = in[ids[p]*d + perm[j]]: the same values as k_gather_soa from the permuted
// SoA copy, read from the row-major input, whose d coordinates of a point share a cache line
template <typename T>
__global__ void k_gather_rows(const T *__restrict__ in, const uint32_t *__restrict__ ids, uint32_t n,
                              uint32_t d, DimPerm perm, T *__restrict__ xs) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const T *row = in + (size_t)ids[p] * d;
  for (uint32_t j = 0; j < d; j++) xs[(size_t)j * n + p] = row[perm.v[j]];
}

// bits[w] bit l = (src[64 w + l] != 0), for the ids below n (the last word's bits past n are 0)
__global__ void k_pack_bits(const uint8_t *__restrict__ src, uint32_t n, uint64_t *__restrict__ bits) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t b = __ballot(i < n && src[i] != 0);
  if ((threadIdx.x & 63u) == 0 && i < n) bits[i >> 6] = b;
}

// Per active query (sorted position p): the number of points in its own cell block (radius
// r = its own, or rAll for every query, cells [coord(x-r) rounded down, coord(x+r) rounded up]) from
// the dense cell-start table.  Fewer than K+1 points there means the query cannot succeed
// at this radius: it is marked failed without a distance evaluation.  The per-cell maximum of
// those counts feeds the algorithmic-bytes accounting (each query cell's block once).
// tryR (full-dimensional grids of 3 or more dims): the radius of the ball that would hold `want`
// points at the block's mean density when the block has over 1.3 times as many per ball, else r;
// the direct kernel searches it first (volD = volume of the unit ball): radii are made to hold
// K+1 points in nearly every ball, and in 6-D a ball with 3 times the points has a block of 3 times
// the candidates.  ms per join without / with: 1M skewed 6-D K=32 on 4 indexed dims learned 45.6 /
// 27.4, 200k uniform 6-D K=16 learned 5.5 / 2.8, 2M uniform 6-D K=32 plain 31.4 / 24.7.
// The active flags come as a bitmap by point id (bit q & 63 of word q >> 6): its 1/8 of a byte
// per point stays in the L2 for these reads in sorted order, where a byte per point (10 MB at
// 10M points) made each read a line from beyond it.
template <typename T, typename G, int ND>
__global__ void k_prefilter(const T *__restrict__ xs, uint32_t n, G g, const T *radius, T rAll,
                            const uint32_t *__restrict__ dense, const uint32_t *__restrict__ sortedIds,
                            const uint64_t *activeBits, uint8_t *failed, uint32_t k1,
                            const uint32_t *cellOf, uint32_t *cellMax, uint32_t *flags, T *tryR, float want,
                            float volD) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t lane = threadIdx.x & 63;
  const bool inRange = p < n;
  const uint32_t q = inRange ? sortedIds[p] : 0u;
  const bool active = inRange && !(activeBits && !((activeBits[q >> 6] >> (q & 63u)) & 1ull));
  uint32_t cnt = 0;
  if (active) {
    const T r = radius ? radius[q] : rAll;
    const T eps = (T)g.eps;
    const uint32_t nd = nd_of<ND>(g);
    // per-dim arrays over a constant bound (registers, not private scratch)
    uint32_t lo[nd_cap<ND>()], hi[nd_cap<ND>()], cur[nd_cap<ND>()];
#pragma unroll
    for (uint32_t j = 0; j < nd_cap<ND>(); j++) {
      if (j >= nd) break;
      const T xj = xs[(size_t)j * n + p];  // cell-sorted copy: the query's own coordinates, coalesced
      lo[j] = cell_coord<T>(next_down(xj - r), (T)g.minArr[j], eps, g.nCells[j]);
      hi[j] = cell_coord<T>(next_up(xj + r), (T)g.minArr[j], eps, g.nCells[j]);
      cur[j] = lo[j];
    }
    if (ND == 1) {
      cnt = dense[g.keyBase + hi[0] + 1] - dense[g.keyBase + lo[0]];
    } else {
      // four rows along dim 1 at a time, their eight reads in flight together (the table has at
      // most 2^28 entries)
      const uint32_t m1 = nd > 1 ? (uint32_t)g.mult[1] : 0u;
      const uint32_t l1 = nd > 1 ? lo[1] : 0u, h1 = nd > 1 ? hi[1] : 0u;
      do {
        const uint32_t base = (uint32_t)row_base<ND>(g, cur);  // (of row l1)
        for (uint32_t c = 0; c <= h1 - l1; c += 4) {
          uint32_t b[4], e[4];
#pragma unroll
          for (uint32_t u = 0; u < 4; u++) {
            const uint32_t at = base + (c + u <= h1 - l1 ? c + u : c) * m1;
            b[u] = dense[at + lo[0]];
            e[u] = dense[at + hi[0] + 1];
          }
#pragma unroll
          for (uint32_t u = 0; u < 4; u++) cnt += c + u <= h1 - l1 ? e[u] - b[u] : 0u;
        }
      } while (next_row<ND, 2>(cur, lo, hi, nd));
    }
    if (tryR) {
      float est = (float)cnt * volD;  // points of the ball at the block's density
      const float reach = (float)(r / eps);
#pragma unroll
      for (uint32_t j = 0; j < nd_cap<ND>(); j++)
        if (j < nd) est *= reach / (float)(hi[j] - lo[j] + 1u);
      tryR[q] = est > 1.3f * want ? r * (T)powf(want / est, 1.0f / (float)nd) : r;
    }
  }
  if (cellMax) {
    // cellOf is non-decreasing in p, so a cell's lanes are one run of the wave: the run's
    // maximum is gathered into its first lane (each lane takes the maximum over the next
    // 1, 2, 4, ... lanes of its own cell), which issues the run's only atomic
    const uint32_t c = inRange ? cellOf[p] : 0xFFFFFFFFu;
    uint32_t m = active ? cnt : 0u;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t mo = __shfl_down(m, o, 64);
      const uint32_t co = __shfl_down(c, o, 64);
      if (lane + o < 64 && co == c && mo > m) m = mo;
    }
    const uint32_t cPrev = __shfl_up(c, 1, 64);
    if (inRange && m && (lane == 0 || cPrev != c)) atomicMax(&cellMax[c], m);
  }
  if (!inRange) return;
  if (!active) {
    flags[p] = 0;
  } else if (cnt < k1) {
    failed[q] = 1;
    flags[p] = 0;
  } else {
    flags[p] = 1;
  }
}

// sum over cells of cellMax (candidate points of each active query cell's block) and the
// number of active query cells; out[0] += points, out[1] += cells.  Grid-stride per thread
// over 16-byte vectors (cellMax comes from an aligned allocation), then a wave reduction and
// one pair of atomics per block.
__global__ __launch_bounds__(256) void k_cell_bytes(const uint32_t *cellMax, uint32_t ncell,
                                                    unsigned long long *out) {
  unsigned long long sp = 0, sc = 0;
  const uint32_t stride = gridDim.x * blockDim.x, gid = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t nv = ncell / 4;
  const uint4 *v4 = reinterpret_cast<const uint4 *>(cellMax);
  for (uint32_t i = gid; i < nv; i += stride) {
    const uint4 v = v4[i];
    sp += (unsigned long long)v.x + (unsigned long long)v.y + (unsigned long long)v.z +
          (unsigned long long)v.w;
    sc += (v.x ? 1ull : 0ull) + (v.y ? 1ull : 0ull) + (v.z ? 1ull : 0ull) + (v.w ? 1ull : 0ull);
  }
  for (uint32_t c = 4 * nv + gid; c < ncell; c += stride) {
    const uint32_t v = cellMax[c];
    sp += v;
    sc += v ? 1ull : 0ull;
  }
  for (int o = 32; o > 0; o >>= 1) {
    sp += __shfl_xor(sp, o, 64);
    sc += __shfl_xor(sc, o, 64);
  }
  // the block's four wave sums, then one pair of atomics per block (every wave adding to the
  // same two counters serialised them)
  __shared__ unsigned long long ws[2][4];
  const uint32_t w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    ws[0][w] = sp;
    ws[1][w] = sc;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned long long bp = ws[0][0] + ws[0][1] + ws[0][2] + ws[0][3];
    const unsigned long long bc = ws[1][0] + ws[1][1] + ws[1][2] + ws[1][3];
    if (bp || bc) {
      atomicAdd(out, bp);
      atomicAdd(out + 1, bc);
    }
  }
}

// cellOf[p] = compacted cell index of sorted position p (inclusive scan of boundary flags - 1)
__global__ void k_cell_of(const uint32_t *flags, const uint32_t *pos, uint32_t n, uint32_t *cellOf) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  cellOf[p] = pos[p] + flags[p] - 1;
}

__global__ void k_active_flags(const uint32_t *sortedIds, const uint8_t *failed, uint32_t n,
                               uint32_t *flags) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  flags[p] = failed ? (uint32_t)failed[sortedIds[p]] : 1u;
}

__global__ void k_compact_active(const uint32_t *sortedIds, const uint32_t *flags,
                                 const uint32_t *pos, uint32_t n, uint32_t *act) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  if (flags[p]) act[pos[p]] = sortedIds[p];
}

// ------------------------------------------------------------------ checksum
constexpr uint32_t SUM_CHUNK = 4096;
// one block per chunk of SUM_CHUNK rows: coalesced copy to LDS, then lane 0 adds in row order (100k
// rows: 47 us with 8 values read before every 8 additions, now 33)
__global__ __launch_bounds__(256) void k_sum_chunks(const double *rowSum, uint32_t n, double *partial) {
  __shared__ __align__(16) double buf[SUM_CHUNK];
  const uint64_t lo = (uint64_t)blockIdx.x * SUM_CHUNK;
  if (lo >= n) return;
  const uint32_t cnt = (uint32_t)(lo + SUM_CHUNK < n ? SUM_CHUNK : n - lo);
  for (uint32_t i = threadIdx.x; i < cnt; i += blockDim.x) buf[i] = rowSum[lo + i];
  __syncthreads();
  if (threadIdx.x == 0) {
    partial[blockIdx.x] = ordered_sum(buf, cnt, 0.0);
  }
}
// Per-row sums in entry order.  A block stages ROWS consecutive rows (one contiguous range of
// the table) in LDS with coalesced loads, then thread r sums row r from LDS.
// 16 KB of rows per block: 8 blocks (32 waves) per CU overlap their loads and sums (32 KB:
// 0.57 ms per 10M x 65 table, 16 KB: 0.45 ms)
constexpr uint32_t SUM_LDS_BYTES = 16384;
template <typename T>
__global__ __launch_bounds__(256) void k_row_sums(const T *__restrict__ dists, uint32_t n, uint32_t k1,
                                                  uint32_t rowsPerBlock, double *rowSum) {
  __shared__ T buf[SUM_LDS_BYTES / sizeof(T)];
  const uint64_t r0 = (uint64_t)blockIdx.x * rowsPerBlock;
  if (r0 >= n) return;
  const uint32_t rows = (uint32_t)((n - r0) < rowsPerBlock ? (n - r0) : rowsPerBlock);
  const T *src = dists + r0 * k1;
  const uint32_t cnt = rows * k1;
  // eight independent loads in flight per thread before their LDS stores
  constexpr uint32_t U = 8;
  for (uint32_t i0 = threadIdx.x; i0 < cnt; i0 += U * 256u) {
    T v[U];
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
      const uint32_t i = i0 + u * 256u;
      v[u] = i < cnt ? src[i] : (T)0;
    }
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
      const uint32_t i = i0 + u * 256u;
      if (i < cnt) buf[i] = v[u];
    }
  }
  __syncthreads();
  for (uint32_t r = threadIdx.x; r < rows; r += blockDim.x) {
    const T *row = buf + (size_t)r * k1;
    double s = 0.0;
    for (uint32_t e = 0; e < k1; e++) {
      const T d = row[e];
      const T sq = d * d;
      s += (double)sq;
    }
    rowSum[r0 + r] = s;
  }
}

// fallback for rows longer than the LDS stage
template <typename T>
__global__ void k_row_sums_direct(const T *__restrict__ dists, uint32_t n, uint32_t k1, double *rowSum) {
  const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  const T *row = dists + (size_t)r * k1;
  double s = 0.0;
  for (uint32_t e = 0; e < k1; e++) {
    const T d = row[e];
    const T sq = d * d;
    s += (double)sq;
  }
  rowSum[r] = s;
}

// one block: the chunks' sums in order, SUM_CHUNK at a time through LDS (2442 chunks: 45 us reading
// global memory 16 at a time, now 18)
__global__ __launch_bounds__(256) void k_sum_final(const double *partial, uint32_t m, double *out) {
  __shared__ __align__(16) double buf[SUM_CHUNK];
  double s = 0.0;
  for (uint32_t c0 = 0; c0 < m; c0 += SUM_CHUNK) {
    const uint32_t cnt = m - c0 < SUM_CHUNK ? m - c0 : SUM_CHUNK;
    __syncthreads();
    for (uint32_t c = threadIdx.x; c < cnt; c += 256) buf[c] = partial[c0 + c];
    __syncthreads();
    if (threadIdx.x == 0) s = ordered_sum(buf, cnt, s);
  }
  if (threadIdx.x == 0) *out = s;
}

}  // namespace

// ------------------------------------------------------------------ host launchers
template <typename T>
void cell_keys_u32(const T *x, uint32_t n, const typename GridOf<T>::type &g, uint32_t *keys,
                   uint32_t *ids, hipStream_t s) {
  if (n) k_cell_keys<T, uint32_t><<<(n + 255) / 256, 256, 0, s>>>(x, n, g, keys, ids);
}
template <typename T>
void cell_keys_u64(const T *x, uint32_t n, const typename GridOf<T>::type &g, uint64_t *keys,
                   uint32_t *ids, hipStream_t s) {
  if (n) k_cell_keys<T, uint64_t><<<(n + 255) / 256, 256, 0, s>>>(x, n, g, keys, ids);
}
void boundary_flags_u32(const uint32_t *keys, uint32_t n, uint32_t sb, uint32_t *flags, hipStream_t s) {
  if (n) k_boundary_flags<uint32_t><<<(n + 255) / 256, 256, 0, s>>>(keys, n, sb, flags);
}
void boundary_flags_u64(const uint64_t *keys, uint32_t n, uint32_t *flags, hipStream_t s) {
  if (n) k_boundary_flags<uint64_t><<<(n + 255) / 256, 256, 0, s>>>(keys, n, 0u, flags);
}
void compact_cells_u32(const uint32_t *keys, const uint32_t *flags, const uint32_t *pos,
                       uint32_t n, uint32_t sb, uint64_t *cellKeys, uint32_t *cellStart, hipStream_t s) {
  if (n) k_compact_cells<uint32_t><<<(n + 255) / 256, 256, 0, s>>>(keys, flags, pos, n, sb, cellKeys, cellStart);
}
void compact_cells_u64(const uint64_t *keys, const uint32_t *flags, const uint32_t *pos,
                       uint32_t n, uint64_t *cellKeys, uint32_t *cellStart, hipStream_t s) {
  if (n) k_compact_cells<uint64_t><<<(n + 255) / 256, 256, 0, s>>>(keys, flags, pos, n, 0u, cellKeys, cellStart);
}
template <typename T>
void gather_soa(const T *x, const uint32_t *ids, uint32_t n, uint32_t d, T *xs, hipStream_t s) {
  if (n) k_gather_soa<T><<<(n + 255) / 256, 256, 0, s>>>(x, ids, n, d, xs);
}
template <typename T>
void gather_rows(const T *in, const uint32_t *ids, uint32_t n, uint32_t d, const DimPerm &perm, T *xs,
                 hipStream_t s) {
  if (n) k_gather_rows<T><<<(n + 255) / 256, 256, 0, s>>>(in, ids, n, d, perm, xs);
}
void gather_u32(const uint32_t *src, const uint32_t *idx, uint32_t n, uint32_t *dst, hipStream_t s) {
  if (n) k_gather_u32<<<(n + 255) / 256, 256, 0, s>>>(src, idx, n, dst);
}
void pack_bits(const uint8_t *src, uint32_t n, uint64_t *bits, hipStream_t s) {
  if (n) k_pack_bits<<<(n + 255) / 256, 256, 0, s>>>(src, n, bits);
}
template <typename T>
void prefilter(const T *xs, uint32_t n, const typename GridOf<T>::type &g, const T *radius,
               T rAll, const uint32_t *dense, const uint32_t *sortedIds, const uint64_t *activeBits,
               uint8_t *failed, uint32_t k1, const uint32_t *cellOf, uint32_t *cellMax,
               uint32_t *flags, T *tryR, float want, hipStream_t s) {
  if (!n) return;
  using G = typename GridOf<T>::type;
  const dim3 grid((n + 255) / 256), block(256);
  float volD = (g.nd & 1) ? 2.0f : 3.14159265f;  // V_1 = 2, V_2 = pi, V_m = V_{m-2} 2 pi / m
  for (uint32_t m = (g.nd & 1) ? 3 : 4; m <= g.nd; m += 2) volD *= 2.0f * 3.14159265f / (float)m;
  switch (g.nd) {
    case 1: k_prefilter<T, G, 1><<<grid, block, 0, s>>>(xs, n, g, radius, rAll, dense, sortedIds, activeBits, failed, k1, cellOf, cellMax, flags, tryR, want, volD); break;
    case 2: k_prefilter<T, G, 2><<<grid, block, 0, s>>>(xs, n, g, radius, rAll, dense, sortedIds, activeBits, failed, k1, cellOf, cellMax, flags, tryR, want, volD); break;
    case 3: k_prefilter<T, G, 3><<<grid, block, 0, s>>>(xs, n, g, radius, rAll, dense, sortedIds, activeBits, failed, k1, cellOf, cellMax, flags, tryR, want, volD); break;
    case 4: k_prefilter<T, G, 4><<<grid, block, 0, s>>>(xs, n, g, radius, rAll, dense, sortedIds, activeBits, failed, k1, cellOf, cellMax, flags, tryR, want, volD); break;
    case 5: k_prefilter<T, G, 5><<<grid, block, 0, s>>>(xs, n, g, radius, rAll, dense, sortedIds, activeBits, failed, k1, cellOf, cellMax, flags, tryR, want, volD); break;
    case 6: k_prefilter<T, G, 6><<<grid, block, 0, s>>>(xs, n, g, radius, rAll, dense, sortedIds, activeBits, failed, k1, cellOf, cellMax, flags, tryR, want, volD); break;
    default: k_prefilter<T, G, 0><<<grid, block, 0, s>>>(xs, n, g, radius, rAll, dense, sortedIds, activeBits, failed, k1, cellOf, cellMax, flags, tryR, want, volD); break;
  }
}
void cell_bytes(const uint32_t *cellMax, uint32_t ncell, unsigned long long *out, hipStream_t s) {
  if (ncell) {
    const uint32_t blocks = (ncell / 4 + 255) / 256 + 1;
    k_cell_bytes<<<blocks < 2048 ? blocks : 2048, 256, 0, s>>>(cellMax, ncell, out);
  }
}
void cell_of(const uint32_t *flags, const uint32_t *pos, uint32_t n, uint32_t *cellOf, hipStream_t s) {
  if (n) k_cell_of<<<(n + 255) / 256, 256, 0, s>>>(flags, pos, n, cellOf);
}

void active_flags(const uint32_t *sortedIds, const uint8_t *failed, uint32_t n, uint32_t *flags,
                  hipStream_t s) {
  if (n) k_active_flags<<<(n + 255) / 256, 256, 0, s>>>(sortedIds, failed, n, flags);
}
void compact_active(const uint32_t *sortedIds, const uint32_t *flags, const uint32_t *pos,
                    uint32_t n, uint32_t *act, hipStream_t s) {
  if (n) k_compact_active<<<(n + 255) / 256, 256, 0, s>>>(sortedIds, flags, pos, n, act);
}

template <typename T>
void row_sums(const T *dists, uint32_t n, uint32_t k1, double *rowSum, hipStream_t s) {
  if (!n) return;
  const uint32_t rpb = (uint32_t)(SUM_LDS_BYTES / sizeof(T) / k1);
  if (rpb >= 1) {
    const uint32_t rows = rpb < 256 ? rpb : 256;
    k_row_sums<T><<<(n + rows - 1) / rows, 256, 0, s>>>(dists, n, k1, rows, rowSum);
  } else {
    k_row_sums_direct<T><<<(n + 255) / 256, 256, 0, s>>>(dists, n, k1, rowSum);
  }
}

void sum_rows(const double *rowSum, uint32_t n, double *partial, double *out, hipStream_t s) {
  const uint32_t m = (n + SUM_CHUNK - 1) / SUM_CHUNK;
  if (m) k_sum_chunks<<<m, 256, 0, s>>>(rowSum, n, partial);
  k_sum_final<<<1, 256, 0, s>>>(partial, m, out);
}

#define INST(T)                                                                                \
  template void cell_keys_u32<T>(const T *, uint32_t, const GridOf<T>::type &, uint32_t *,      \
                                 uint32_t *, hipStream_t);                                     \
  template void cell_keys_u64<T>(const T *, uint32_t, const GridOf<T>::type &, uint64_t *,      \
                                 uint32_t *, hipStream_t);                                     \
  template void gather_soa<T>(const T *, const uint32_t *, uint32_t, uint32_t, T *, hipStream_t); \
  template void gather_rows<T>(const T *, const uint32_t *, uint32_t, uint32_t, const DimPerm &, T *, \
                               hipStream_t);                                                   \
  template void row_sums<T>(const T *, uint32_t, uint32_t, double *, hipStream_t);          \
  template void prefilter<T>(const T *, uint32_t, const GridOf<T>::type &, const T *, T,      \
                             const uint32_t *, const uint32_t *, const uint64_t *, uint8_t *, \
                             uint32_t, const uint32_t *, uint32_t *, uint32_t *, T *, float, hipStream_t);
INST(float)
INST(double)
#undef INST

}  // namespace knn
