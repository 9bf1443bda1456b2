// direct.hip -- the direct range kernel for gfx950: the exact top-(K+1) of each query from the
// grid cells around it, one wavefront per query.
//
// Replaces kernel.cu:61-225 (range query over the adjacent cells), the pair buffer and the two
// thrust::stable_sort_by_key of GPU.cu:1629-1634, and the host top-k of GPU.cu:3610-3704.
//
// Ranking: FP64 key = sum_j ((double)c_j - (double)q_j)^2, ties by point id.
// Success: at least K+1 candidates with key <= Tq = r^2 (1 - 2^-20).  Every point with key <= Tq
// lies within r of the query in each indexed dim, hence inside the streamed block, so a success
// is the exact global top-(K+1).  The reference's FP32 test (kernel.cu:130-147) differs from
// this only for candidates within 2^-20 of eps.
//
// Work unit: a chunk of up to 64 consecutive active queries (cell order; a tile in a batched
// group), taken from a queue by a persistent wave.  The chunk's geometry is set up with lane =
// query, then the queries run in turn with lane = candidate:
//   stream   the query's own block (rows narrowed to the chords of its ball, cells cut to its
//            slab), 64 candidates a round, several rounds' loads in flight.  With up to 2 indexed
//            dims the rows are looked up for the whole chunk at once (64 queries share the memory
//            round trip), and a query whose block holds more points than it needs is first tried
//            at the radius that should hold K+1 + 3 sqrt(K+1) of them; if that fails it runs
//            again at its full radius.  A block of up to 192 points goes to the selection straight
//            from its rounds; otherwise a candidate whose T sum is within the bound of the current
//            threshold enters an LDS list of sorted positions (ballot order).  A full list is
//            tightened: a histogram of its keys gives an edge that still holds K+1 of them, which
//            becomes the threshold.
//   select   the items (FP64 keys in registers) are counted into DR_NB equal buckets of [0,
//            threshold] in LDS; an exclusive scan turns the counts into slots (a counting sort),
//            each item is ranked against the items of its own bucket, and the first K+1 go to the
//            row.
// The bucket of a key is the low word of key * (DR_NB - 1) / threshold + 1.5 * 2^52 (one fused
// multiply-add): a monotone function of the key, so bucket order is key order.
// A query whose list does not fit (thousands of equal keys) goes to the overflow kernel
// (range.hip).
//
// What bounds it: VALU issue in 2-D (72 % of the issue slots at 4 waves per SIMD; about 350 vector
// instructions per query at K = 64, failed searches included, of which the selection is about 150).  One query per wave needs no
// tile of queries around a shared union of blocks, so few queries left in a pass still fill the
// chip, and each candidate is loaded only for queries whose ball may hold it.  Against the kernel
// before it (a tile-wide histogram pass, then a second pass over each query's sub-block; the
// collect kernel with 5 or more indexed dims), range-kernel ms per join on one MI355X, same rows:
// 10M mixed 2-D K=64 learned 11.4 / 7.9, plain 21.5 / 10.9; 5M skewed 4-D K=32 learned 30.1 /
// 10.8; 2M uniform 6-D K=32 plain 38.7 / 20.4; 1M skewed 6-D on 4 dims K=32 learned 107 / 16.9 (there
// on a grid over all 6 dims).
// 128 registers (4 waves per SIMD): 96 (5 waves) spills and loses 25 % in 2-D.
#include "knn_range.h"

#ifndef KNN_DIRECT_PART
#define KNN_DIRECT_PART 0
#endif

namespace knn {
namespace {

constexpr double DR_MAGIC = 6755399441055744.0;  // 1.5 * 2^52

// lane mask of a condition (the builtin keeps a comparison's mask as it is)
__device__ __forceinline__ uint64_t ballot64(bool c) { return __builtin_amdgcn_ballot_w64(c); }
__device__ __forceinline__ uint32_t mbcnt64(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
__device__ __forceinline__ uint32_t rl(uint32_t v, uint32_t i) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)i);
}

__device__ __forceinline__ uint32_t dr_bucket(double key, double scale) {
  return (uint32_t)__double_as_longlong(__builtin_fma(key, scale, DR_MAGIC));
}

// Correctly rounded square roots of sums of squares.  FP32: the hardware root is within one
// ulp, and its neighbours are tested with Tuckerman's criterion (y is the rounded root of s iff
// y (y - u) < s <= y (y + u), evaluated by fused multiply-adds); sums below 2^-96 take the
// library function, whose scaling the fused products need there.
__device__ __forceinline__ float root_of(float s) {
  const float y = __builtin_amdgcn_sqrtf(s);
  const float yd = __int_as_float(__float_as_int(y) - 1), yu = __int_as_float(__float_as_int(y) + 1);
  const float rd = __builtin_fmaf(-yd, y, s), ru = __builtin_fmaf(-yu, y, s);
  float v = rd <= 0.0f ? yd : y;
  v = ru > 0.0f ? yu : v;
  return v;
}
__device__ __forceinline__ bool root_small(float s) { return s < 0x1p-96f && s != 0.0f; }
__device__ __forceinline__ bool root_small(double) { return false; }
__device__ __forceinline__ double root_of(double s) { return sqrt(s); }

// waves per SIMD the register budget is set for: 4 (128 registers), 2 for the largest lists
constexpr int waves_per_simd(int h) { return h <= 4 ? 4 : 2; }
// Windows of 64 candidates that a chunk's row tables cover, and those kept in registers: the last
// two of the 8 at H = 4 live in LDS (1 KB, within the 10 KB of 16 waves per CU).  All 8 in
// registers spill 18 of the 128: range-kernel ms, 10M mixed 2-D K=64 learned 8.9 / 8.1 and plain
// 13.5 / 11.6, 3M mixed K=128 learned 6.8 / 6.4 (6.3 now), 3M uniform K=200 plain 9.1 /
// 8.7.
constexpr uint32_t windows(int h) { return h >= 4 ? 8 : 4; }
constexpr uint32_t reg_windows(int h) { return h == 4 ? 6 : windows(h); }
// LDS: DR_NB bucket counters and 64 dummies, H * 64 sorted (key, id) slots and four sentinels, a
// list of positions, and with a row table DR_RMAX words and the last windows per query of a chunk
constexpr uint32_t list_cap(int h, bool tab) { return h * 64 + (tab && h == 3 ? 128 : 256); }
constexpr size_t lds_bytes(int h, bool tab) {
  return ((size_t)(DR_NB + 64) * 4 + (size_t)(h * 64 + 4) * 12 + (size_t)list_cap(h, tab) * 4 +
          (tab ? 64 * DR_RMAX * 4 + 64 * (windows(h) - reg_windows(h)) * 8 : 0) + 15) & ~(size_t)15;
}

// Rounds of a selection of NR rounds that hold 64 items each, whatever its item count: 1..4 rounds
// take counts above 64 (NR - 1), 8 rounds take every count above 256.
constexpr int full_rounds(int nr) { return nr <= 4 ? nr - 1 : 4; }

template <int N>
struct IntC {
  static constexpr int value = N;
};

// T sum of a candidate with fused multiply-adds, within 2^-19 of the key (the filter; the
// reported distance uses the unfused sum)
template <typename T, int D>
__device__ __forceinline__ T filter_sum(const T *c, const T *q) {
  T s = (T)0;
#pragma unroll
  for (int j = 0; j < D; j++) {
    const T df = c[j] - q[j];
    if constexpr (std::is_same<T, float>::value)
      s = __builtin_fmaf(df, df, s);
    else
      s = s + df * df;
  }
  return s;
}

// Row ranges of the block [lo, hi] (wave-uniform), lane = row rb + lane: the row's cells within
// the query's ball (chord of r2 in dim 0), pB = first sorted position, len = its point count
// (0 past the last row or outside the ball).  Fewer than 2^18 rows: the row's coordinates come
// from float quotients ((t + 1/2) / span lies at least 1/(2 span) from an integer, more than the
// error of the reciprocal and the product).
template <typename T, int D, int ND, typename G>
__device__ __forceinline__ void ball_rows(const JoinArgs &a, const G &g, const CellGeo<T> *geo, const uint32_t *lo,
                                          const uint32_t *hi, const T *q, const double *qd, T r, double r2, uint32_t R,
                                          uint32_t rr, uint32_t &pB, uint32_t &len) {
  pB = 0;
  len = 0;
  uint32_t t = rr < R ? rr : R - 1u;
  uint64_t rowBase = g.keyBase;
  double d2 = r2;
  const double invr2 = r > (T)0 ? 1.0 / ((double)r * (double)r) : 0.0;
#pragma unroll
  for (int j = 1; j < ND; j++) {
    const uint32_t span = hi[j] - lo[j] + 1u;
    uint32_t c = t;
    if (j < ND - 1) {
      const uint32_t h = (uint32_t)(((float)t + 0.5f) * __builtin_amdgcn_rcpf((float)span));
      c = t - h * span;
      t = h;
    }
    c += lo[j];
    rowBase += (uint64_t)c * g.mult[j];
    d2 -= cell_gap2<T>(geo[j], c, qd[j]);
  }
  if (rr < R && d2 >= 0.0) {
    uint32_t l, u;
    cell_span<T>(geo[0], q[0], half_chord(d2, r, invr2), l, u);
    l = l > lo[0] ? l : lo[0];
    u = u < hi[0] ? u : hi[0];
    if (l <= u) {
      uint32_t pE;
      row_range(a, rowBase, l, u, pB, pE);
      len = pE - pB;
    }
  }
}

template <typename T, int D, int ND, int H, bool SETS, typename G>
__global__ __launch_bounds__(64, waves_per_simd(H)) void k_direct(JoinArgs a, G g0, GeoArgs<T, (ND > 0 ? ND : 1)> ga) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr bool TAB = ND == 1 || ND == 2;
  // rounds of a stream loaded together (ms per join with one more / one less: 1M skewed 6-D K=32 on 4
  // dims 22.2 / 23.1 / 25.5, 2M uniform 6-D K=32 plain 23.1 / 22.9 / 23.7, 300k uniform 8-D K=16
  // - / 15.0 / 16.9, 3M uniform 4-D K=32 plain 8.2 / 8.3 / 8.5)
  constexpr int PR = TAB ? 2 : (D <= 4 ? 4 : (D <= 8 ? 3 : 1));
  constexpr uint32_t RM = ND == 1 ? 1 : DR_RMAX;
  constexpr uint32_t NW = windows(H), NWR = reg_windows(H);
  constexpr uint32_t CAP = list_cap(H, TAB);  // list slots
  constexpr uint32_t ROOM = CAP - 64u * PR;
  uint32_t *hist = reinterpret_cast<uint32_t *>(smem);  // DR_NB counters, 64 dummies
  double *skey = reinterpret_cast<double *>(hist + DR_NB + 64);  // H * 64 sorted keys, 4 sentinels
  uint32_t *sid = reinterpret_cast<uint32_t *>(skey + H * 64 + 4);
  uint32_t *list = sid + H * 64 + 4;
  uint32_t *rowB = list + CAP;  // TAB: position offsets of the chunk's rows, DR_RMAX per query
  uint64_t *winH = reinterpret_cast<uint64_t *>(rowB + 64 * DR_RMAX);  // TAB: windows from NWR on
  uint32_t *segB = sid, *segX = sid + 64;  // a stream's segment tables (the sorted ids come later)
  const uint32_t lane = threadIdx.x;
  const T *__restrict__ xs = reinterpret_cast<const T *>(a.xs);
  const T *__restrict__ x = reinterpret_cast<const T *>(a.x);
  const size_t n = a.n;
  const char *xsb[D];
#pragma unroll
  for (int j = 0; j < D; j++) xsb[j] = reinterpret_cast<const char *>(xs + (size_t)j * n);
  const char *idb = reinterpret_cast<const char *>(a.sortedIds);
  auto load1 = [&](uint32_t p, T (&c)[D]) {
    if constexpr (ND > 0) {
      const uint32_t off = p * (uint32_t)sizeof(T);
#pragma unroll
      for (int j = 0; j < D; j++) c[j] = *reinterpret_cast<const T *>(xsb[j] + off);
    } else {
#pragma unroll
      for (int j = 0; j < D; j++) c[j] = xs[(size_t)j * n + p];
    }
  };
  auto load_id = [&](uint32_t p) -> uint32_t {
    if constexpr (ND > 0) return *reinterpret_cast<const uint32_t *>(idb + p * 4u);
    return a.sortedIds[p];
  };
  uint32_t Q;
  const uint32_t NT = work_count(a, TAB ? 1u : 4u, ND >= 1 && ND <= 4, Q);
  WaveTally tally;
  bool first = true;
  for (;;) {
    const uint32_t t = next_tile(a.tileCounter, NT, a.tileRanges, lane, first);
    if (t >= NT) break;
    first = false;
    const uint2 tl = work_tile(a, t, Q);
    const uint32_t nq = tl.y;
    const uint32_t qL = tile_query(a, tl, lane < nq ? lane : 0u);
    TileCtx<G> C;
    if constexpr (SETS) {
      C = tile_ctx<G>(a, g0, tl);
    } else {
      C.k1 = a.k1;
      C.idBase = 0;
      C.rowAdj = 0;
    }
    const G &g = SETS ? C.g : g0;
    const uint32_t nd = nd_of<ND>(g);
    const uint32_t K1 = C.k1;
    const T eps = (T)g.eps;
    // ---- chunk set-up (lane = query)
    T qcL[D];
#pragma unroll
    for (int j = 0; j < D; j++) qcL[j] = x[(size_t)j * n + qL];
    const T rL = a.radius ? reinterpret_cast<const T *>(a.radius)[qL] : (T)a.radiusAll;
    // rows of the query's block, concatenated: candidate f of row k (X_k <= f < X_{k+1}) sits at
    // f + rowB[k]; the row of f is counted from a bitmap of the starts (bit X_k - 1, so that the
    // bits below a lane's own are the starts at or before its candidate)
    uint32_t RL = 0, totL = 0;
    uint64_t winL[NWR] = {};
    wave_lds_sync();
    T rs = rL;  // the radius searched first
    if (!TAB && !SETS && a.tryRadius) rs = reinterpret_cast<const T *>(a.tryRadius)[qL];
    if constexpr (TAB) {
      const double q1 = ND >= 2 ? (double)qcL[ND - 1] : 0.0;
      auto lookup = [&](T rr) {
        const CellGeo<T> g0 = SETS ? cell_geo<T, G>(g, 0) : ga.c[0], g1 = SETS ? cell_geo<T, G>(g, ND - 1) : ga.c[ND - 1];
        uint32_t l0s, h0s, l1 = 0, h1 = 0, cells = 0;
        cell_span_fast<T>(g0, qcL[0], rr, l0s, h0s);
        if (ND >= 2) cell_span_fast<T>(g1, qcL[ND - 1], rr, l1, h1);
        RL = 0;
        totL = 0;
#pragma unroll
        for (uint32_t w = 0; w < NWR; w++) winL[w] = 0;
#pragma unroll
        for (uint32_t w = NWR; w < NW; w++) winH[lane * (NW - NWR) + w - NWR] = 0;
        const bool fits = h1 - l1 < RM;
        const double r2 = (double)rr * (double)rr * (1.0 + 0x1p-15), invr2 = rr > (T)0 ? 1.0 / ((double)rr * (double)rr) : 0.0;
        // ranges of row k (none past the block or outside the ball): start, point count
        auto range_of = [&](uint32_t k, uint32_t &pB, uint32_t &len) {
          const uint32_t c = l1 + k;
          pB = 0;
          len = 0;
          if (!(fits && c <= h1)) return;
          double d2 = r2;
          uint32_t l = l0s, u = h0s;
          if (ND >= 2) {
            d2 -= cell_gap2<T>(g1, c, q1);
            if (!(d2 >= 0.0)) return;
            cell_span_fast<T>(g0, qcL[0], half_chord(d2, rr, invr2), l, u);
            l = l > l0s ? l : l0s;
            u = u < h0s ? u : h0s;
          }
          if (l <= u) {
            const uint64_t rowBase = g.keyBase + (ND >= 2 ? (uint64_t)c * g.mult[ND - 1] : 0ull);
            pB = a.denseStart[rowBase + l];
            len = a.denseStart[rowBase + u + 1] - pB;
            cells += u - l + 1u;
          }
        };
        auto append = [&](uint32_t pB, uint32_t len) {
          if (!len) return;
          rowB[lane * DR_RMAX + RL] = pB - totL;
          const uint32_t b = totL - 1u;
#pragma unroll
          for (int w = 0; w < (int)NWR; w++)
            if (RL && (b >> 6) == (uint32_t)w) winL[w] |= 1ull << (b & 63u);
          if (NWR < NW && RL && (b >> 6) >= NWR && (b >> 6) < NW)
            winH[lane * (NW - NWR) + (b >> 6) - NWR] |= 1ull << (b & 63u);
          RL++;
          totL += len;
        };
        // two rows a step (one with a.lookupRows = 1): their table reads are in flight together
#pragma unroll 1
        for (uint32_t k = 0; k < RM; k += a.lookupRows) {
          uint32_t pA, nA, pB = 0, nB = 0;
          range_of(k, pA, nA);
          if (ND >= 2 && a.lookupRows == 2u) range_of(k + 1u, pB, nB);
          append(pA, nA);
          append(pB, nB);
        }
        if (totL > 64u * NW || !fits) RL = 0;
        else if (RL == 0) RL = 1;  // nothing in the block: no candidates, no rows to look up
        return cells;
      };
      const T del0 = SETS ? cell_geo<T, G>(g, 0).del : ga.c[0].del;
      const T del1 = SETS ? cell_geo<T, G>(g, ND - 1).del : ga.c[ND - 1].del;
      if (a.denseStart && !g.sb && del0 <= (T)0.25 && del1 <= (T)0.25) {
        const uint32_t cells = lookup(rL);
        if constexpr (ND == D) {
          // a block with more points than needed: search the radius that holds about
          // K+1 + 3 sqrt(K+1) points at the block's density first
          const float want = (float)K1 + 3.0f * sqrtf((float)K1) + 2.0f;
          const float reach = (float)(rL / eps);
          const float vol = (ND == 2 ? 3.14159265f * reach : 2.0f) * reach / (float)cells;
          const float est = (float)totL * vol;
          if (est > 1.1f * want) rs = rL * (T)(ND == 2 ? sqrtf(want / est) : want / est);
          if (ballot64(rs < rL)) lookup(rs);
        }
      }
    }
    const double TqL = (double)rs * (double)rs * (1.0 - 0x1p-20);
    const double scL = TqL > 0.0 ? (double)(DR_NB - 1) / TqL : 0.0;
    const uint64_t shrunk = ballot64(rs < rL);
    wave_lds_sync();
    uint64_t okMask = 0, ovMask = 0;
    unsigned long long seen = 0;

    for (uint32_t i = 0; i < nq; i++) {
      T qi[D];
      double qd[D];
#pragma unroll
      for (int j = 0; j < D; j++) {
        qi[j] = readlane<T>(qcL[j], (int)i);
        qd[j] = (double)qi[j];
      }
      const uint32_t qid = rl(qL, i);
      double Tc = readlane<double>(TqL, (int)i);
      double sc = readlane<double>(scL, (int)i);
      T Fc = Num<T>::bound(Tc);
      uint32_t M = 0;
      bool ovf = false;
      auto clear_hist = [&]() {
        reinterpret_cast<uint4 *>(hist)[lane] = make_uint4(0u, 0u, 0u, 0u);
        wave_lds_sync();
      };

      // a full list: the threshold drops to a bucket edge that still holds K+1 keys, and the
      // items beyond it leave the list
      auto tighten = [&](uint32_t room) {
        wave_lds_sync();
        clear_hist();
        for (uint32_t e0 = 0; e0 < M; e0 += 64) {
          const uint32_t e = e0 + lane;
          T c[D];
          load1(list[e < M ? e : 0u], c);
          const double key = fp64_key<D, T>(c, qd);
          if (e < M && key <= Tc) atomicAdd(&hist[dr_bucket(key, sc)], 1u);
        }
        wave_lds_sync();
        const uint4 h = reinterpret_cast<const uint4 *>(hist)[lane];
        const uint32_t inc = wave_incl_sum(h.x + h.y + h.z + h.w, lane);
        const uint64_t at = ballot64(inc >= K1);
        if (at == 0) {
          ovf = true;
          return;
        }
        uint32_t cum = inc - (h.x + h.y + h.z + h.w);
        uint32_t b = 4u * lane;
        if (cum + h.x < K1) {
          cum += h.x;
          b++;
          if (cum + h.y < K1) {
            cum += h.y;
            b++;
            if (cum + h.z < K1) b++;
          }
        }
        const uint32_t bs = rl(b, (uint32_t)__builtin_ctzll(at));
        const double Tn = readfirst<double>(((double)bs + 0.5) / sc * (1.0 + 0x1p-40));
        if (Tn < Tc) {
          Tc = Tn;
          sc = readfirst<double>((double)(DR_NB - 1) / Tc);
          Fc = Num<T>::bound(Tc);
        }
        uint32_t M2 = 0;
        for (uint32_t e0 = 0; e0 < M; e0 += 64) {
          const uint32_t e = e0 + lane;
          const uint32_t p = list[e < M ? e : 0u];
          T c[D];
          load1(p, c);
          const double key = fp64_key<D, T>(c, qd);
          const bool keep = e < M && key <= Tc;
          const uint64_t m = ballot64(keep);
          wave_lds_sync();
          if (keep) list[M2 + mbcnt64(m)] = p;
          M2 += (uint32_t)__popcll(m);
          wave_lds_sync();
        }
        M = M2;
        if (M > room) ovf = true;
      };

      // NR rounds of candidates (lanes from cnt[u] on hold none): loads, the filter, the list
      auto push = [&](auto nr, const uint32_t *pv, const uint32_t *cnt) {
        constexpr int NR = decltype(nr)::value;
        T cv[NR][D];
#pragma unroll
        for (int u = 0; u < NR; u++) load1(pv[u], cv[u]);
#pragma unroll
        for (int u = 0; u < NR; u++)
#pragma unroll
          for (int j = 0; j < D; j++) asm volatile("" ::"v"(cv[u][j]));
#pragma unroll
        for (int u = 0; u < NR; u++) {
          const bool near = (lane < cnt[u]) & (filter_sum<T, D>(cv[u], qi) <= Fc);
          const uint64_t m = ballot64(near);
          const uint32_t at = M + mbcnt64(m);
          if (near) list[at] = pv[u];
          M += (uint32_t)__popcll(m);
        }
      };

      const uint32_t Ri = TAB ? rl(RL, i) : 0u;
      // ---- select: m items' keys in registers, counting sort, rank within the bucket
      auto fin = [&](auto nr, const uint32_t *pv, uint32_t m, bool direct) {
        constexpr int NR = decltype(nr)::value;
        constexpr int FULL = full_rounds(NR);
        clear_hist();
        T cv[NR][D];
        uint32_t id[NR];
#pragma unroll
        for (int u = 0; u < NR; u++) {
          load1(pv[u], cv[u]);
          id[u] = load_id(pv[u]);
        }
#pragma unroll
        for (int u = 0; u < NR; u++) {
#pragma unroll
          for (int j = 0; j < D; j++) asm volatile("" ::"v"(cv[u][j]));
          asm volatile("" ::"v"(id[u]));
        }
        double key[NR];
        T ss[NR];
        bool in[NR];
        uint32_t b[NR], sl[NR], st[NR];
#pragma unroll
        for (int u = 0; u < NR; u++) {
          key[u] = fp64_key<D, T>(cv[u], qd);
          ss[u] = Num<T>::template sq<D>(cv[u], qi);
          in[u] = (key[u] <= Tc) & (u < FULL || 64u * u + lane < m);
          b[u] = in[u] ? dr_bucket(key[u], sc) : DR_NB + lane;
        }
        if (direct) {
          uint32_t got = 0;
#pragma unroll
          for (int u = 0; u < NR; u++) got += (uint32_t)__popcll(ballot64(in[u]));
          if (got < K1) return;  // fails at this radius
        }
#pragma unroll
        for (int u = 0; u < NR; u++) sl[u] = atomicAdd(&hist[b[u]], 1u);
        wave_lds_sync();
        const uint4 h = reinterpret_cast<const uint4 *>(hist)[lane];
        const uint32_t inc = wave_incl_sum(h.x + h.y + h.z + h.w, lane);
        const uint32_t total = rl(inc, 63);
        if (total < K1) return;  // fails at this radius
        const uint32_t e0 = inc - (h.x + h.y + h.z + h.w), e1 = e0 + h.x, e2 = e1 + h.y, e3 = e2 + h.z;
        const uint32_t hm = max(max(h.x, h.y), max(h.z, h.w));
        reinterpret_cast<uint4 *>(hist)[lane] = make_uint4(e0, e1, e2, e3);
        wave_lds_sync();
#pragma unroll
        for (int u = 0; u < NR; u++) st[u] = hist[b[u]];
#pragma unroll
        for (int u = 0; u < NR; u++) asm volatile("" ::"v"(st[u]));
#pragma unroll
        for (int u = 0; u < NR; u++) {
          if (in[u]) {
            skey[st[u] + sl[u]] = key[u];
            sid[st[u] + sl[u]] = id[u];
          }
          st[u] = in[u] ? st[u] : K1;  // lanes without an item rank nothing (K1 <= total)
        }
        if (lane < 4u) skey[total + lane] = __builtin_inf();
        wave_lds_sync();
        // The slots from an item's bucket on hold its bucket's items, then larger keys: the
        // number of smaller keys among the first four is its rank within a bucket of up to four.
        // Equal keys (more matches than the items' own) and larger buckets take the loop below.
        uint32_t rk[NR];
        uint32_t eq = 0, own = 0;
#pragma unroll
        for (int u = 0; u < NR; u++) {
          const double k0 = skey[st[u]], k1 = skey[st[u] + 1], k2 = skey[st[u] + 2], k3 = skey[st[u] + 3];
          rk[u] = st[u] + (k0 < key[u] ? 1u : 0u) + (k1 < key[u] ? 1u : 0u) + (k2 < key[u] ? 1u : 0u) + (k3 < key[u] ? 1u : 0u);
          own += (uint32_t)__popcll(ballot64(in[u]));
          eq += (uint32_t)__popcll(ballot64(in[u] & (k0 == key[u]))) + (uint32_t)__popcll(ballot64(in[u] & (k1 == key[u]))) +
                (uint32_t)__popcll(ballot64(in[u] & (k2 == key[u]))) + (uint32_t)__popcll(ballot64(in[u] & (k3 == key[u])));
        }
        if (eq != own || ballot64(hm > 4u)) {
#pragma unroll
          for (int u = 0; u < NR; u++) {
            if (in[u]) {
              uint32_t r = st[u];
              const uint32_t w1 = b[u] == DR_NB - 1 ? total : hist[b[u] + 1];
              for (uint32_t v = st[u]; v < w1; v++) r += kless(skey[v], sid[v], key[u], id[u]) ? 1u : 0u;
              rk[u] = r;
            }
          }
        }
        char *rowI = reinterpret_cast<char *>(a.outIds + C.row(qid));
        char *rowD = reinterpret_cast<char *>(reinterpret_cast<T *>(a.outDists) + C.row(qid));
#pragma unroll
        for (int u = 0; u < NR; u++) {
          T y = root_of(ss[u]);
          if (ballot64(in[u] & root_small(ss[u]))) y = sqrt(ss[u]);
          if (in[u] & (rk[u] < K1)) {
            *reinterpret_cast<int32_t *>(rowI + rk[u] * 4u) = (int32_t)(id[u] - C.idBase);
            *reinterpret_cast<T *>(rowD + rk[u] * (uint32_t)sizeof(T)) = y;
          }
        }
        okMask |= 1ull << i;
      };
      // ---- stream
      for (uint32_t tryFull = (TAB ? Ri != 0u : ((shrunk >> i) & 1ull) != 0ull) ? 0u : 1u;; tryFull = 1u) {
      if (TAB && !tryFull) {
        const uint32_t tot = rl(totL, i);
        seen += tot;
        uint32_t run = i * DR_RMAX;  // first row of the window: its slot in rowB
        auto tabled = [&](auto nr, auto wb) {
          constexpr int NR = decltype(nr)::value, W0 = decltype(wb)::value;
          uint32_t pv[NR], cnt[NR];
#pragma unroll
          for (int u = 0; u < NR; u++) {
            uint64_t w;
            if constexpr (W0 + NR > (int)NWR) {
              const uint64_t wm = W0 + u < (int)NWR ? winL[W0 + u < (int)NWR ? W0 + u : 0]
                                                    : winH[i * (NW - NWR) + (uint32_t)(W0 + u) - NWR];
              const uint32_t from = W0 + u < (int)NWR ? i : 0u;
              w = (uint64_t)rl((uint32_t)wm, from) | ((uint64_t)rl((uint32_t)(wm >> 32), from) << 32);
            } else {
              const uint64_t wm = winL[W0 + u];
              w = (uint64_t)rl((uint32_t)wm, i) | ((uint64_t)rl((uint32_t)(wm >> 32), i) << 32);
            }
            const uint32_t k = run + mbcnt64(w);
            run += (uint32_t)__popcll(w);
            const uint32_t f0 = 64u * (W0 + u), fi = f0 + lane;
            cnt[u] = u < NR - 1 ? 64u : tot - f0;
            const uint32_t f = u == NR - 1 ? (fi < tot ? fi : tot - 1u) : fi;
            pv[u] = f + rowB[k];
          }
          if (W0 == 0 && NR <= 3)
            fin(nr, pv, tot, true);
          else
            push(nr, pv, cnt);
        };
        if (NW > 4 && tot > 256u) {
          constexpr int B = NW > 4 ? 4 : 0;
          tabled(IntC<4>(), IntC<0>());
          if (tot <= 320u) tabled(IntC<1>(), IntC<B>());
          else if (tot <= 384u) tabled(IntC<2>(), IntC<B>());
          else if (tot <= 448u) tabled(IntC<3>(), IntC<B>());
          else tabled(IntC<4>(), IntC<B>());
        } else if (tot > 192u) tabled(IntC<4>(), IntC<0>());
        else if (tot > 128u) tabled(IntC<3>(), IntC<0>());
        else if (tot > 64u) tabled(IntC<2>(), IntC<0>());
        else if (tot) tabled(IntC<1>(), IntC<0>());
      } else {
        const T r = readlane<T>(TAB || tryFull ? rL : rs, (int)i);
        auto group = [&](const uint32_t (&pv)[PR], const bool (&)[PR], uint32_t f0, uint32_t tot) {
          if (ovf) return;
          if (M > ROOM) {
            tighten(ROOM);
            if (ovf) return;
          }
          const uint32_t left = tot - f0;
          uint32_t cnt[PR];
#pragma unroll
          for (int u = 0; u < PR; u++) cnt[u] = left > 64u * u ? left - 64u * u : 0u;
          if (PR == 1 || left <= 64u) push(IntC<1>(), pv, cnt);
          else if (PR == 2 || left <= 128u) push(IntC<(PR >= 2 ? 2 : 1)>(), pv, cnt);
          else push(IntC<PR>(), pv, cnt);
        };
        Tc = (double)r * (double)r * (1.0 - 0x1p-20);
        sc = readfirst<double>(Tc > 0.0 ? (double)(DR_NB - 1) / Tc : 0.0);
        Fc = Num<T>::bound(Tc);
        M = 0;
        CellGeo<T> geo[ND > 0 ? ND : 1];
#pragma unroll
        for (uint32_t j = 0; j < (uint32_t)ND; j++) geo[j] = SETS ? cell_geo<T, G>(g, j) : ga.c[j];
        uint32_t lo[nd_cap<ND>()], hi[nd_cap<ND>()];
#pragma unroll
        for (uint32_t j = 0; j < nd_cap<ND>(); j++) {
          if (j >= nd) break;
          const T xj = pick_t<T, D>(qi, j);
          if constexpr (ND > 0) {
            cell_span<T>(geo[j], xj, r, lo[j], hi[j]);
            lo[j] = readfirst<uint32_t>(lo[j]);
            hi[j] = readfirst<uint32_t>(hi[j]);
            continue;
          }
          lo[j] = readfirst<uint32_t>(cell_coord<T>(next_down(xj - r), (T)g.minArr[j], eps, g.nCells[j]));
          hi[j] = readfirst<uint32_t>(cell_coord<T>(next_up(xj + r), (T)g.minArr[j], eps, g.nCells[j]));
        }
        const double r2 = (double)r * (double)r * (1.0 + 0x1p-15);
        const bool cut = (ND > 0 && ND < D) && g.sb && hi[0] - lo[0] < SLAB_MAX_SPAN;
        const uint64_t R = block_rows<ND>(g, lo, hi);
        const uint64_t RS = cut ? R * (uint64_t)(hi[0] - lo[0] + 1) : R;
        uint32_t sql = 0, sqh = 0;
        if (cut) {
          const T xq = pick_t<T, D>(qi, nd);
          sql = readfirst<uint32_t>(slab_q<T>(next_down(xq - r), g));
          sqh = readfirst<uint32_t>(slab_q<T>(next_up(xq + r), g));
        }
        uint32_t mine = 0;
        for (uint64_t rb = 0; rb < RS; rb += 64) {
          uint32_t pB, len;
          if (cut)
            seg_batch<T, D, ND, G>(a, g, lo, hi, nd >= 2, qd, r2, RS, rb + lane, sql, sqh, xs + (size_t)nd * n, pB, len);
          else if (ND > 0 && R < (1ull << 18))
            ball_rows<T, D, ND, G>(a, g, geo, lo, hi, qi, qd, r, r2, (uint32_t)R, (uint32_t)rb + lane, pB, len);
          else
            row_batch<T, D, ND, G>(a, g, lo, hi, nd >= 2, qd, r2, R, rb + lane, pB, len);
          mine += len;
          stream_segments<PR>(pB, len, lane, segB, segX, a.segCapLog2, group);
        }
        seen += rl(wave_incl_sum(mine, lane), 63);
      }
      wave_lds_sync();
      if (!ovf && M > 64u * H) tighten(64u * H);

      if (!ovf && M >= K1) {
        auto from_list = [&](auto nr) {
          constexpr int NR = decltype(nr)::value;
          uint32_t pv[NR];
#pragma unroll
          for (int u = 0; u < NR; u++) {
            const uint32_t e = 64u * u + lane;
            pv[u] = list[u < full_rounds(NR) ? e : (e < M ? e : 0u)];
          }
          fin(nr, pv, M, false);
        };
        if (M <= 64u) from_list(IntC<1>());
        else if (M <= 128u) from_list(IntC<2>());
        else if (H == 3 || M <= 192u) from_list(IntC<3>());
        else if (H == 4 || M <= 256u) from_list(IntC<(H >= 4 ? 4 : 1)>());
        else from_list(IntC<(H >= 8 ? 8 : 1)>());
      }
      if (tryFull || ovf || ((okMask >> i) & 1ull) || !((shrunk >> i) & 1ull)) break;
      }
      if (ovf) ovMask |= 1ull << i;
      wave_lds_sync();
    }
    const bool okL = (okMask >> lane) & 1ull, ovL = (ovMask >> lane) & 1ull;
    if (lane < nq) {
      if (ovL)
        a.overflow[qL] = 1;
      else
        a.failed[qL] = okL ? 0 : 1;
    }
    if (lane == 0 && ovMask) atomicAdd(a.overflowCount, (uint32_t)__popcll(ovMask));
    tally.fails += nq - (uint32_t)__popcll(okMask | ovMask);
    tally.bytes += (unsigned long long)nq * 8ull + (unsigned long long)__popcll(okMask) * K1 * (4ull + sizeof(T));
    tally.cand += seen;
  }
  flush_tally(a, tally, lane);
}

template <typename T, int D, int ND, typename G>
void launch_nd(const JoinArgs &a, const G &g, hipStream_t s) {
  constexpr bool tab = ND == 1 || ND == 2;
  GeoArgs<T, (ND > 0 ? ND : 1)> ga{};
  if (!a.sets)
    for (int j = 0; j < (ND > 0 ? ND : 1); j++) ga.c[j] = cell_geo<T, G>(g, (uint32_t)j);
  auto run = [&](auto hc) {
    constexpr int H = decltype(hc)::value;
    // persistent grid: the waves the registers admit on 256 CUs (the caller's for batched groups)
    const uint32_t grid = a.sets ? a.ntiles : 256u * 4u * (uint32_t)waves_per_simd(H);
    if constexpr (std::is_same<T, float>::value) {
      if (a.sets) {
        k_direct<T, D, ND, H, true, G><<<grid, 64, lds_bytes(H, tab), s>>>(a, g, ga);
        return;
      }
    }
    k_direct<T, D, ND, H, false, G><<<grid, 64, lds_bytes(H, tab), s>>>(a, g, ga);
  };
  if (a.k1 <= direct_k1(3)) run(IntC<3>());
  else if (a.k1 <= direct_k1(4)) run(IntC<4>());
  else if constexpr (ND == 0 || D <= 4) run(IntC<8>());
  else launch_nd<T, D, 0, G>(a, g, s);  // (one build for the rare long rows of many dims)
}

}  // namespace

template <typename T, int D>
void direct_launch(const JoinArgs &a, const typename GridOf<T>::type &g, hipStream_t s) {
  using G = typename GridOf<T>::type;
  if ((uint64_t)a.n * sizeof(T) > 0xffffffffull) {
    launch_nd<T, D, 0, G>(a, g, s);  // 64-bit addressing throughout
    return;
  }
  switch (g.nd) {
    case 1: launch_nd<T, D, 1, G>(a, g, s); return;
    case 2: if constexpr (D >= 2) launch_nd<T, D, 2, G>(a, g, s); return;
    case 3: if constexpr (D >= 3) launch_nd<T, D, 3, G>(a, g, s); return;
    case 4: if constexpr (D >= 4) launch_nd<T, D, 4, G>(a, g, s); return;
    case 5: if constexpr (D >= 5) launch_nd<T, D, 5, G>(a, g, s); return;
    case 6: if constexpr (D >= 6) launch_nd<T, D, 6, G>(a, g, s); return;
    default: launch_nd<T, D, 0, G>(a, g, s); return;
  }
}

#define DR_INST(T, D) template void direct_launch<T, D>(const JoinArgs &, const GridOf<T>::type &, hipStream_t);
#if KNN_DIRECT_PART < 8
#define KNN_DR_T float
#else
#define KNN_DR_T double
#endif
DR_INST(KNN_DR_T, 2 * (KNN_DIRECT_PART % 8) + 1)
DR_INST(KNN_DR_T, 2 * (KNN_DIRECT_PART % 8) + 2)

}  // namespace knn
