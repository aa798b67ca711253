// Brute-force radius search (LinearKNNSearch::find_radius,
// linear_search.rs:89-108): every row with distance <= radius, in index order.
//
// Euclidian searches take one sweep of FP64 matrix tiles (further down).  The
// others, and what that form leaves over, take two passes
// over the same tiled distance block as the kNN scan: `count`
// tallies matches per (query, segment); an exclusive scan turns the tallies
// into CSR offsets; `fill` recomputes the block and writes each query's
// matches of a tile in index order at its running offset.  When every query
// block scans all rows (one segment: large query sets, such as DBSCAN's
// search of every row), one `capped` pass instead writes each query's
// matches, in index order, to a slot of kCap entries while counting all of
// them; a compaction kernel moves the slots to CSR order, and the queries
// with more than kCap matches are searched again as a subset with the two
// passes.  The lists are the same either way.  A row is tested
// with a conservative bound on the sum first and then exactly on the
// finalised distance (sqrt / identity / powf(1/p)), so the decision is the
// reference's `d <= radius`.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "common.hpp"
#include "metric.hpp"
#include "mfma64.hpp"
#include "tile.hpp"

namespace sc {
namespace {

constexpr int QT = kTileQ;
constexpr int RT = kTileR;
constexpr int NT = kTileThreads;

// Kernel modes: count matches per (query, segment); fill them at CSR
// offsets; or (one segment) write them to a kCap-entry slot per query while
// counting all.
constexpr int kCount = 0, kFill = 1, kCapped = 2;
constexpr int64_t kCap = 256;
// Largest capped buffer (index and distance slots) one search may take.
constexpr double kCapBytes = 1024.0 * 1024.0 * 1024.0;

// DIST: the matches' distances are written too (their LDS buffer, 32 KB,
// would otherwise cost occupancy).
template <typename T, int M, int MODE, bool DIST>
__global__ __launch_bounds__(NT) void radius_kernel(const T* __restrict__ refs, int64_t n, int ld, int d,
                                                    const T* __restrict__ queries, int64_t q,
                                                    double p, double radius, double sum_bound,
                                                    int64_t seg_len, int nseg,
                                                    uint64_t* __restrict__ counts,
                                                    int64_t* __restrict__ out_idx,
                                                    double* __restrict__ out_dist, int64_t cap) {
  __shared__ TileSmem<T> sm;
  __shared__ double dbuf[DIST ? QT : 1][DIST ? RT : 1];
  __shared__ uint32_t mask[QT][RT / 32];
  const int tid = threadIdx.x;
  const int tq = tid >> 5;
  const int tr = tid & 31;
  const int64_t q0 = static_cast<int64_t>(blockIdx.x) * QT;
  const int seg = blockIdx.y;
  const int64_t r_begin = static_cast<int64_t>(seg) * seg_len;
  const int64_t r_end = min(n, r_begin + seg_len);
  for (int e = tid; e < QT * (RT / 32); e += NT) (&mask[0][0])[e] = 0u;
  const int64_t my_q = q0 + tid;
  uint64_t run = 0;
  if (MODE == kFill && tid < QT && my_q < q) run = counts[static_cast<size_t>(my_q) * nseg + seg];

  for (int64_t t0 = r_begin; t0 < r_end; t0 += RT) {
    double acc[4][4];
    tile_sums<T, M>(sm, acc, refs, t0, r_end, queries, q0, q, ld, d, p);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int qi = tq * 4 + i;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int rl = tr + 32 * j;
        if (q0 + qi < q && t0 + rl < r_end && acc[i][j] <= sum_bound) {
          const double dv = finalize<M>(acc[i][j], p);
          if (dv <= radius) {
            if constexpr (DIST) dbuf[qi][rl] = dv;
            atomicOr(&mask[qi][rl >> 5], 1u << (rl & 31));
          }
        }
      }
    }
    __syncthreads();
    if (tid < QT && my_q < q) {
      for (int w = 0; w < RT / 32; ++w) {
        uint32_t bits = mask[tid][w];
        mask[tid][w] = 0u;
        if (MODE == kCount) {
          run += static_cast<uint64_t>(__popc(bits));
          continue;
        }
        while (bits) {
          const int b = __builtin_ctz(bits);
          bits &= bits - 1;
          const int rl = w * 32 + b;
          if (MODE == kFill) {
            out_idx[run] = t0 + rl;
            if constexpr (DIST) out_dist[run] = dbuf[tid][rl];
          } else if (run < static_cast<uint64_t>(cap)) {
            const size_t o = static_cast<size_t>(my_q) * static_cast<size_t>(cap) + run;
            out_idx[o] = t0 + rl;
            if constexpr (DIST) out_dist[o] = dbuf[tid][rl];
          }
          ++run;
        }
      }
    }
  }
  if (MODE != kFill && tid < QT && my_q < q) counts[static_cast<size_t>(my_q) * nseg + seg] = run;
}

// Slots of the capped pass to CSR order: query i with at most cap matches
// moves them to offsets[i] (one wavefront per query); queries with more are
// left to their own search.
__global__ void radius_compact_kernel(const int64_t* __restrict__ cidx,
                                      const double* __restrict__ cdist, int64_t cap,
                                      const uint64_t* __restrict__ counts,
                                      const uint64_t* __restrict__ offsets, int64_t q,
                                      int64_t* __restrict__ out_idx, double* __restrict__ out_dist) {
  const int lane = threadIdx.x & 63;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * (blockDim.x / 64) + (threadIdx.x >> 6);
  if (i >= q) return;
  const uint64_t c = counts[i];
  if (c > static_cast<uint64_t>(cap)) return;
  const uint64_t o = offsets[i];
  const size_t base = static_cast<size_t>(i) * static_cast<size_t>(cap);
  for (uint64_t j = lane; j < c; j += 64) {
    out_idx[o + j] = cidx[base + j];
    if (out_dist) out_dist[o + j] = cdist[base + j];
  }
}

// Rows list[0 .. m) of src (stride ld), gathered into dst.
template <typename T>
__global__ void gather_rows_kernel(const T* __restrict__ src, int ld,
                                   const int64_t* __restrict__ list, int64_t m,
                                   T* __restrict__ dst) {
  const int64_t total = m * ld;
  for (int64_t e = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; e < total;
       e += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t r = e / ld;
    dst[e] = src[list[r] * ld + (e - r * ld)];
  }
}

// ---- Euclidian searches on FP64 matrix instructions (mfma64.hpp) ----
//
//   sweep    128 x 128 tiles; the rows whose lower bound on the sum passes
//            the radius go to a list per (query, piece) in row order.  The
//            (query tile, row tile) pairs, query tiles outermost, are dealt
//            to the workgroups in contiguous runs; a piece is the part of a
//            run inside one query tile.  A candidate whose upper bound is
//            inside the radius too is a match; the others make their list
//            unsure.
//   resolve  a workgroup per query: the exact distances of the unsure lists'
//            candidates, whose matches move to the front of the list, and the
//            query's count (kUnresolved when a list overflowed or the query's
//            norm is out of the bound's range).
//   emit     the matches to their CSR place, with their distances.
// Queries whose lists overflowed are swept once more into lists of the sizes
// that the first sweep counted; norms out of range take the count and fill
// passes.
// One sweep takes the place of a count and a fill pass, and an MFMA per four
// dimensions that of three vector instructions per dimension and pair.  With
// many matches the sweep's time goes to appending them (5,000 queries x
// 100,000 x 16 f32: 0.41 ms with 20 matches each, 1.01 with 1,417; the two
// passes 2.7), so matches are neither counted nor summed twice: 0.12 ms for
// 7.1 million of them, whole calls 581 and 2,387 us with 20 matches, 7,500 and
// 9,700 with 1,417 (sweep and two passes).  Summing every candidate to count it, by
// one wavefront per query, and sending queries past 65,536 entries to the two
// passes made 10 queries x 1,000,000 x 8 f64 with 50,000 matches each 3,300 us;
// they take 661 now and 683 with the two passes.
constexpr uint32_t kUnresolved = 0xffffffffu;
constexpr uint64_t kNoPlace = ~uint64_t(0);
// Lists of a sweep: room for every pair, or 256 MiB in all (but 256 entries
// per query).
constexpr int64_t kListTotal = int64_t(1) << 26;
constexpr int64_t kListMin = 256;
constexpr int64_t kSweepQueries = int64_t(1) << 19;  // per sweep
constexpr uint64_t kSecondMax = uint64_t(1) << 31;   // entries of a second sweep
// Fewer pairs take the two passes, whose three launches fewer count there (us,
// two passes and sweep): 1.0 M pairs, 1,000 queries x 1,000 x 8 f64, 29 matches
// each: 120 and 131; 100 x 10,000 x 4 f64, 6 to 3,225 matches: 75 to 346 and 75
// to 365; 2.0 M, 50 x 40,000 x 16 f32, 5 to 12,000: 89 to 381 and 79 to 397.  From
// 3.0 M on the sweep is ahead at any number of matches: 212 x 14,151 x 21 f32, 5
// to 3,999: 114 to 506 and 86 to 489; 1,000 x 3,000 x 32 f32, 5 to 886: 140 to 515 and
// 110 to 504; 3 x 1,000,000 x 8 f64, 5 to 50,000: 202 to 363 and 131 to 329.
constexpr double kSweepMinPairs = 3.5e6;

// The candidate lists of a sweep: `lists` per query, each with room for cap
// entries, or (second sweep) from where `starts` says, kNoPlace for the queries
// that take no part.
struct RadiusLists {
  uint32_t* idx;
  uint32_t* count;   // q x lists: candidates, after resolve matches
  uint32_t* unsure;  // q x lists
  const uint64_t* starts;
  int lists;
  int64_t cap;
  __device__ __forceinline__ int64_t at(int64_t qi, int l) const {
    return starts ? static_cast<int64_t>(starts[qi * lists + l]) : (qi * lists + l) * cap;
  }
  __device__ __forceinline__ bool takes(int64_t qi) const { return !starts || starts[qi * lists] != kNoPlace; }
};

// sure: sums up to it are inside the radius.
template <typename T, bool SECOND>
__global__ __launch_bounds__(kMT, 2) void radius_sweep_kernel(
    const T* __restrict__ rows, int64_t n, int ld, int d, const double* __restrict__ y2m,
    const T* __restrict__ queries, int64_t q, const double* __restrict__ x2m, Bound64 bd,
    double bound, double sure, int64_t tiles, int64_t per, RadiusLists out) {
  __shared__ MSmem sm;
  const MLane ml;
  const int64_t nqt = (q + kMQ - 1) / kMQ;
  int64_t pos = static_cast<int64_t>(blockIdx.x) * per;
  const int64_t end = min(pos + per, nqt * tiles);
  while (pos < end) {
    const int64_t qt = pos / tiles;
    const int64_t tb = pos - qt * tiles;
    const int64_t te = min(tiles, tb + (end - pos));
    const int list = static_cast<int>(blockIdx.x - qt * tiles / per);
    const int64_t q0 = qt * kMQ;
    pos += te - tb;
    double th[2], x2[2];
    int64_t at[2] = {0, 0};
    uint32_t cnt[2] = {0u, 0u}, uns[2] = {0u, 0u};  // the same in all four lanes of a column
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t qi = q0 + ml.query_of(j);
      x2[j] = qi < q && (!SECOND || out.takes(qi)) ? x2m[qi] : INFINITY;
      th[j] = x2[j] < INFINITY ? acc_threshold(bd, bound, x2[j]) : -INFINITY;
      if (x2[j] < INFINITY) at[j] = out.at(qi, list);
    }
    if (SECOND && !__syncthreads_or(x2[0] < INFINITY || x2[1] < INFINITY)) continue;
    mfma64_sweep<T, false>(sm, rows, n, ld, d, y2m, queries, q, q0, 0, tb, te,
                           [&](int64_t t, MAcc& acc, int par) {
      tile_hits(ml, acc, th, sm.y2[par], [&](int i, int j, int v, int rl, bool hit, uint64_t m) {
        m &= ml.column();
        const uint32_t c = cnt[j] + __popcll(m & ml.below());
        if (hit && (SECOND || static_cast<int64_t>(c) < out.cap))
          out.idx[at[j] + c] = static_cast<uint32_t>(t * kMR + rl);
        cnt[j] += __popcll(m);
        if (!SECOND) {
          const double u = sum_upper(bd, acc[i][j][v] + x2[j], x2[j] + sm.y2[par][rl]);
          uns[j] += __popcll(__ballot(hit && !(u <= sure)) & ml.column());
        }
      });
    });
    if (!SECOND) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int64_t qi = q0 + ml.query_of(j);
        if (ml.lg == 0 && qi < q) {
          out.count[qi * out.lists + list] = cnt[j];
          out.unsure[qi * out.lists + list] = uns[j];
        }
      }
    }
    __syncthreads();  // the sweep's LDS is staged anew
  }
}

// total: the candidates of a query whose lists overflowed, else 0.
constexpr int kResolveThreads = 256;
template <typename T>
__global__ __launch_bounds__(kResolveThreads) void radius_resolve_kernel(
    const T* __restrict__ rows, int ld, const T* __restrict__ queries, int64_t q, double radius,
    RadiusLists ls, uint32_t* __restrict__ matches, uint32_t* __restrict__ total) {
  __shared__ uint32_t s_sum[kResolveThreads / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int64_t qi = blockIdx.x;
  uint32_t* count = ls.count + qi * ls.lists;
  if (!ls.takes(qi)) {
    if (threadIdx.x == 0) matches[qi] = kUnresolved;
    return;
  }
  // the sum over the workgroup's threads, in thread 0
  auto sum = [&](uint32_t v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    if (lane == 0) s_sum[wave] = v;
    __syncthreads();
    if (threadIdx.x == 0)
      for (int w = 1; w < waves; ++w) v += s_sum[w];
    return v;
  };
  if (!ls.starts) {
    uint32_t all = 0;
    bool over = false;
    for (int l = threadIdx.x; l < ls.lists; l += blockDim.x) {
      const uint32_t c = count[l];
      all += c;
      over = over || static_cast<int64_t>(c) > ls.cap;
    }
    if (__syncthreads_or(over)) {
      // the counts stay those of the sweep: a second one goes by them
      all = sum(all);
      if (threadIdx.x == 0) {
        matches[qi] = kUnresolved;
        total[qi] = all;
      }
      return;
    }
  }
  uint32_t found = 0;
  for (int l0 = 64 * wave; l0 < ls.lists; l0 += 64 * waves) {  // lane = list
    const bool in = l0 + lane < ls.lists;
    uint32_t c = in ? count[l0 + lane] : 0u;
    uint64_t open = __ballot(in && ls.unsure[qi * ls.lists + l0 + lane] != 0u);
    while (open) {  // the whole wavefront takes one list
      const int src = __builtin_ctzll(open);
      open &= open - 1;
      const uint32_t m = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(c), src));
      uint32_t* mine = ls.idx + ls.at(qi, l0 + src);
      uint32_t kept = 0;
      for (uint32_t e0 = 0; e0 < m; e0 += 64) {
        bool match = false;
        uint32_t row = 0;
        if (e0 + lane < m) {
          row = mine[e0 + lane];
          match = __builtin_sqrt(exact_sum<T, kEuclid>(queries + qi * ld, rows + static_cast<int64_t>(row) * ld, ld)) <= radius;
        }
        // to the front: no entry that is still to be read is overwritten
        const uint64_t b = __ballot(match);
        if (match) mine[kept + __popcll(b & ((uint64_t(1) << lane) - 1))] = row;
        kept += static_cast<uint32_t>(__popcll(b));
      }
      if (lane == src) {
        c = kept;
        count[l0 + lane] = kept;
      }
    }
    found += c;
  }
  found = sum(found);
  if (threadIdx.x != 0) return;
  matches[qi] = found;
  if (total) total[qi] = 0u;
}

__global__ void radius_mark_kernel(const uint32_t* __restrict__ list,
                                   const uint32_t* __restrict__ list_n,
                                   uint32_t* __restrict__ matches) {
  const uint32_t n = *list_n;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    matches[list[i]] = kUnresolved;
}

// Where the lists of a second sweep start: base[qi] (kNoPlace: takes no part),
// one list after another.  One wavefront per query.
__global__ __launch_bounds__(64) void radius_starts_kernel(const uint64_t* __restrict__ base,
                                                           const uint32_t* __restrict__ count, int lists,
                                                           uint64_t* __restrict__ starts) {
  const int lane = threadIdx.x;
  const int64_t qi = blockIdx.x;
  uint64_t at = base[qi];
  for (int l0 = 0; l0 < lists; l0 += 64) {
    const uint32_t c = l0 + lane < lists ? count[qi * lists + l0 + lane] : 0u;
    uint32_t inc = c;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t up = __shfl_up(inc, o);
      if (lane >= o) inc += up;
    }
    if (l0 + lane < lists) starts[qi * lists + l0 + lane] = at == kNoPlace ? kNoPlace : at + inc - c;
    if (at != kNoPlace) at += __shfl(inc, 63);
  }
}

// A wavefront takes a query's matches 64 at a time, every gridDim.y-th 64 of
// them (few queries with many matches would leave the chip idle otherwise).
// Its rows go through LDS by whole wavefronts (metric.hpp).
template <typename T>
__global__ __launch_bounds__(64) void radius_emit_kernel(
    const T* __restrict__ rows, int ld, const T* __restrict__ queries, RadiusLists ls,
    const uint32_t* __restrict__ matches, const uint64_t* __restrict__ offsets,
    int64_t* __restrict__ out_idx, double* __restrict__ out_dist, int staged) {
  // the query row (staged), then the lists' starts (lists + 1)
  extern __shared__ __align__(16) unsigned char emit_smem[];
  __shared__ __align__(16) unsigned char tile[kSumTileBytes];
  T* qrow = reinterpret_cast<T*>(emit_smem);
  uint32_t* start = reinterpret_cast<uint32_t*>(qrow + (staged ? ld : 0));
  const int lane = threadIdx.x;
  const int64_t qi = blockIdx.x;
  const uint32_t c = matches[qi];
  if (c == kUnresolved || 64u * blockIdx.y >= c) return;
  if (staged)
    for (int j = lane; j < ld; j += 64) qrow[j] = queries[qi * ld + j];
  uint32_t acc = 0;
  for (int l0 = 0; l0 < ls.lists; l0 += 64) {
    const uint32_t v = l0 + lane < ls.lists ? ls.count[qi * ls.lists + l0 + lane] : 0u;
    uint32_t inc = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t up = __shfl_up(inc, o);
      if (lane >= o) inc += up;
    }
    if (l0 + lane < ls.lists) start[l0 + lane] = acc + inc - v;
    acc += __shfl(inc, 63);
  }
  __syncthreads();
  const uint64_t o = offsets[qi];
  for (uint64_t e0 = 64u * blockIdx.y; e0 < c; e0 += 64u * gridDim.y) {
    const uint32_t e = static_cast<uint32_t>(min(e0 + lane, static_cast<uint64_t>(c) - 1));
    int lo = 0, hi = ls.lists;  // the last list that starts at or below e
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (start[mid] <= e)
        lo = mid;
      else
        hi = mid;
    }
    const uint32_t row = ls.idx[ls.at(qi, lo) + (e - start[lo])];
    const bool mine = e0 + lane < c;
    if (mine) out_idx[o + e] = row;
    if (out_dist) {
      const double sum = staged ? wave_exact_sums<T, kEuclid>(qrow, rows, row, ld, tile)
                                : exact_sum<T, kEuclid>(queries + qi * ld, rows + static_cast<int64_t>(row) * ld, ld);
      if (mine) out_dist[o + e] = __builtin_sqrt(sum);
    }
  }
}

__global__ void radius_zero_kernel(uint32_t* p, int64_t n) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x)
    p[i] = 0u;
}

template <typename T, int M>
int run_radius(const sc_index* ix, const T* dq, int64_t q, double p, double radius,
               sc_radius_result* res, bool want_dist, bool allow_cap, hipStream_t s);

// Queries `over` searched again by the count and fill passes: their lists,
// in the order of `over`.
template <typename T, int M>
int search_subset(const sc_index* ix, const T* dq, const std::vector<int64_t>& over, double p,
                  double radius, sc_radius_result* sub, bool want_dist, hipStream_t s) {
  const int ld = static_cast<int>(ix->ld);
  const int64_t m = static_cast<int64_t>(over.size());
  DevBuf dl, dsub;
  SC_HIP(dl.alloc(sizeof(int64_t) * m, s));
  SC_HIP(hipMemcpyAsync(dl.p, over.data(), sizeof(int64_t) * m, hipMemcpyHostToDevice, s));
  SC_HIP(dsub.alloc(sizeof(T) * m * ld, s));
  const int64_t g = std::min<int64_t>(4096, (m * ld + 255) / 256);
  hipLaunchKernelGGL((gather_rows_kernel<T>), dim3(static_cast<unsigned>(std::max<int64_t>(1, g))),
                     dim3(256), 0, s, dq, ld, dl.as<int64_t>(), m, dsub.as<T>());
  SC_HIP(hipGetLastError());
  return run_radius<T, M>(ix, dsub.as<T>(), m, p, radius, sub, want_dist, false, s);
}

// The Euclidian search for a radius whose bound is in range.
template <typename T>
int run_radius_f64(const sc_index* ix, const T* dq, int64_t q, double radius, double bound,
                   sc_radius_result* res, bool want_dist, hipStream_t s) {
  const int64_t n = static_cast<int64_t>(ix->n);
  const int ld = static_cast<int>(ix->ld), d = static_cast<int>(ix->d);
  const T* rows = static_cast<const T*>(ix->rows);
  const Bound64 bd = bound64<T>(ld);
  // sqrt(S) <= radius for every S up to this, whatever the roundings
  const double sure = radius * radius * (1.0 - 1e-12);
  DevBuf local;
  const double* y2m = nullptr;
  if (int rc = ensure_norms64(const_cast<sc_index*>(ix), local, &y2m, s)) return rc;
  const int64_t nqt = (q + kMQ - 1) / kMQ;
  const int64_t tiles = (n + kMR - 1) / kMR;
  // two workgroups per CU fit; each takes the same number of tiles
  const int64_t per = std::max<int64_t>(1, (nqt * tiles + 511) / 512);
  const int lists = static_cast<int>(std::min<int64_t>((tiles + per - 1) / per + 1, tiles));
  const int64_t entries = std::max(kListMin, kListTotal / q);
  const int64_t cap = std::max<int64_t>(16, std::min<int64_t>(per * kMR, entries / lists));
  const int64_t words = q * lists;
  DevBuf x2m, olist, flags, idx, cnt, mat, tot;
  SC_HIP(x2m.alloc(sizeof(double) * q, s));
  SC_HIP(olist.alloc(sizeof(uint32_t) * q, s));
  SC_HIP(flags.alloc(16, s));
  SC_HIP(idx.alloc(sizeof(uint32_t) * words * cap, s));
  SC_HIP(cnt.alloc(sizeof(uint32_t) * 2 * words, s));  // count | unsure
  SC_HIP(mat.alloc(sizeof(uint32_t) * q, s));
  SC_HIP(tot.alloc(sizeof(uint32_t) * q, s));
  const RadiusLists ls{idx.as<uint32_t>(), cnt.as<uint32_t>(), cnt.as<uint32_t>() + words, nullptr, lists, cap};
  hipLaunchKernelGGL(radius_zero_kernel, dim3(static_cast<unsigned>(std::min<int64_t>(1024, (2 * words + 255) / 256))),
                     dim3(256), 0, s, cnt.as<uint32_t>(), 2 * words);
  hipLaunchKernelGGL(radius_zero_kernel, dim3(1), dim3(64), 0, s, flags.as<uint32_t>(), int64_t{4});
  if (int rc = query_norms64<T>(dq, q, ld, x2m.as<double>(), olist.as<uint32_t>(),
                                flags.as<uint32_t>(), s))
    return rc;
  const dim3 groups(static_cast<unsigned>((nqt * tiles + per - 1) / per));
  const dim3 resolve_threads(static_cast<unsigned>(std::min(kResolveThreads, (lists + 63) / 64 * 64)));
  {
    ProfScope ps("radius_sweep", s);
    hipLaunchKernelGGL((radius_sweep_kernel<T, false>), groups, dim3(kMT), 0, s, rows, n, ld, d, y2m, dq, q,
                       x2m.as<double>(), bd, bound, sure, tiles, per, ls);
    SC_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL(radius_resolve_kernel<T>, dim3(static_cast<unsigned>(q)), resolve_threads, 0, s, rows, ld,
                     dq, q, radius, ls, mat.as<uint32_t>(), tot.as<uint32_t>());
  hipLaunchKernelGGL(radius_mark_kernel, dim3(4), dim3(256), 0, s, olist.as<uint32_t>(),
                     flags.as<uint32_t>(), mat.as<uint32_t>());
  SC_HIP(hipGetLastError());
  std::vector<uint32_t> hm(static_cast<size_t>(q));
  if (int rc = download_staged(hm.data(), mat.p, sizeof(uint32_t) * hm.size(), s)) return rc;
  std::vector<int64_t> over;
  for (int64_t i = 0; i < q; ++i)
    if (hm[i] == kUnresolved) over.push_back(i);
  // the second sweep's lists, and what is left to the two passes
  DevBuf idx2, base2, start2, mat2;
  RadiusLists ls2{};
  std::vector<uint32_t> hm2;
  if (!over.empty()) {
    std::vector<uint32_t> ht(static_cast<size_t>(q));
    if (int rc = download_staged(ht.data(), tot.p, sizeof(uint32_t) * ht.size(), s)) return rc;
    std::vector<uint64_t> base(static_cast<size_t>(q), kNoPlace);
    std::vector<int64_t> rest;
    uint64_t at = 0;
    for (const int64_t i : over) {
      // (no candidates: a norm out of the bound's range)
      if (ht[i] == 0 || at + ht[i] > kSecondMax) {
        rest.push_back(i);
        continue;
      }
      base[i] = at;
      at += ht[i];
    }
    // (lists that do not fit the memory: the two passes)
    if (at > 0 && idx2.alloc(sizeof(uint32_t) * at, s) == hipSuccess) {
      SC_HIP(base2.alloc(sizeof(uint64_t) * q, s));
      SC_HIP(start2.alloc(sizeof(uint64_t) * words, s));
      SC_HIP(mat2.alloc(sizeof(uint32_t) * q, s));
      if (int rc = upload_staged(base2.p, base.data(), sizeof(uint64_t) * q, s)) return rc;
      ls2 = ls;
      ls2.idx = idx2.as<uint32_t>();
      ls2.starts = start2.as<uint64_t>();
      hipLaunchKernelGGL(radius_starts_kernel, dim3(static_cast<unsigned>(q)), dim3(64), 0, s, base2.as<uint64_t>(),
                         cnt.as<uint32_t>(), lists, start2.as<uint64_t>());
      {
        ProfScope ps("radius_sweep", s);
        hipLaunchKernelGGL((radius_sweep_kernel<T, true>), groups, dim3(kMT), 0, s, rows, n, ld, d, y2m, dq, q,
                           x2m.as<double>(), bd, bound, sure, tiles, per, ls2);
      }
      hipLaunchKernelGGL(radius_resolve_kernel<T>, dim3(static_cast<unsigned>(q)), resolve_threads, 0, s, rows,
                         ld, dq, q, radius, ls2, mat2.as<uint32_t>(), static_cast<uint32_t*>(nullptr));
      SC_HIP(hipGetLastError());
      hm2.resize(static_cast<size_t>(q));
      if (int rc = download_staged(hm2.data(), mat2.p, sizeof(uint32_t) * hm2.size(), s)) return rc;
      for (const int64_t i : over)
        if (base[i] != kNoPlace) hm[i] = hm2[i];
      over.swap(rest);
    } else if (at > 0) {
      (void)hipGetLastError();
    }
  }
  if (static_cast<int64_t>(over.size()) == q)
    return run_radius<T, kEuclid>(ix, dq, q, 2.0, radius, res, want_dist, false, s);
  sc_radius_result sub;
  if (!over.empty())
    if (int rc = search_subset<T, kEuclid>(ix, dq, over, 2.0, radius, &sub, want_dist, s)) return rc;
  res->q = static_cast<size_t>(q);
  res->offsets.resize(static_cast<size_t>(q) + 1);
  uint64_t total = 0;
  uint32_t most = 0;  // matches of a query that the lists hold
  size_t next = 0;
  for (int64_t i = 0; i < q; ++i) {
    res->offsets[i] = total;
    if (hm[i] == kUnresolved) {
      total += sub.offsets[next + 1] - sub.offsets[next];
      ++next;
    } else {
      total += hm[i];
      most = std::max(most, hm[i]);
    }
  }
  res->offsets[q] = total;
  res->idx.resize(total);
  if (want_dist) res->dist.resize(total);
  if (total == 0) return SC_OK;
  DevBuf off, oi, od;
  SC_HIP(off.alloc(sizeof(uint64_t) * (q + 1), s));
  if (int rc = upload_staged(off.p, res->offsets.data(), sizeof(uint64_t) * (q + 1), s)) return rc;
  SC_HIP(oi.alloc(sizeof(int64_t) * total, s));
  if (want_dist) SC_HIP(od.alloc(sizeof(double) * total, s));
  // wavefronts for the whole chip, as far as there are matches for them
  const unsigned split = static_cast<unsigned>(
      std::max<int64_t>(1, std::min<int64_t>((int64_t{most} + 63) / 64, (16384 + q - 1) / q)));
  const int staged = want_dist && sizeof(T) * ld <= 32768 ? 1 : 0;
  auto emit = [&](const RadiusLists& l, const DevBuf& m) {
    hipLaunchKernelGGL(radius_emit_kernel<T>, dim3(static_cast<unsigned>(q), split), dim3(64),
                       (staged ? sizeof(T) * ld : 0) + sizeof(uint32_t) * (lists + 1), s, rows, ld, dq, l,
                       m.as<uint32_t>(), off.as<uint64_t>(), oi.as<int64_t>(),
                       want_dist ? od.as<double>() : nullptr, staged);
  };
  emit(ls, mat);
  if (!hm2.empty()) emit(ls2, mat2);
  SC_HIP(hipGetLastError());
  if (int rc = download_staged(res->idx.data(), oi.p, sizeof(int64_t) * total, s)) return rc;
  if (want_dist)
    if (int rc = download_staged(res->dist.data(), od.p, sizeof(double) * total, s)) return rc;
  for (size_t j = 0; j < over.size(); ++j) {
    const uint64_t b = sub.offsets[j], c = sub.offsets[j + 1] - b, o = res->offsets[over[j]];
    std::copy(sub.idx.begin() + b, sub.idx.begin() + b + c, res->idx.begin() + o);
    if (want_dist) std::copy(sub.dist.begin() + b, sub.dist.begin() + b + c, res->dist.begin() + o);
  }
  return SC_OK;
}

// The one-segment search: capped pass, compaction, and the queries past the
// cap searched again (count and fill passes) and merged in.
template <typename T, int M>
int run_radius_capped(const sc_index* ix, const T* dq, int64_t q, double p, double radius,
                      double bound, sc_radius_result* res, bool want_dist, hipStream_t s) {
  const int64_t n = static_cast<int64_t>(ix->n);
  const int ld = static_cast<int>(ix->ld);
  const int64_t nqt = (q + QT - 1) / QT;
  const int64_t tiles = std::max<int64_t>(1, (n + RT - 1) / RT);
  DevBuf cnt, ci, cd;
  SC_HIP(cnt.alloc(sizeof(uint64_t) * q, s));
  SC_HIP(ci.alloc(sizeof(int64_t) * q * kCap, s));
  if (want_dist) SC_HIP(cd.alloc(sizeof(double) * q * kCap, s));
  {
    ProfScope ps("radius_capped", s);
    if (want_dist)
      hipLaunchKernelGGL((radius_kernel<T, M, kCapped, true>), dim3(static_cast<unsigned>(nqt), 1),
                         dim3(NT), 0, s, static_cast<const T*>(ix->rows), n, ld,
                         static_cast<int>(ix->d), dq, q, p, radius, bound, tiles * RT, 1,
                         cnt.as<uint64_t>(), ci.as<int64_t>(), cd.as<double>(), kCap);
    else
      hipLaunchKernelGGL((radius_kernel<T, M, kCapped, false>), dim3(static_cast<unsigned>(nqt), 1),
                         dim3(NT), 0, s, static_cast<const T*>(ix->rows), n, ld,
                         static_cast<int>(ix->d), dq, q, p, radius, bound, tiles * RT, 1,
                         cnt.as<uint64_t>(), ci.as<int64_t>(), nullptr, kCap);
    SC_HIP(hipGetLastError());
  }
  std::vector<uint64_t> hc(static_cast<size_t>(q));
  SC_HIP(hipMemcpyAsync(hc.data(), cnt.p, sizeof(uint64_t) * hc.size(), hipMemcpyDeviceToHost, s));
  SC_HIP(hipStreamSynchronize(s));
  res->q = static_cast<size_t>(q);
  res->offsets.assign(static_cast<size_t>(q) + 1, 0);
  uint64_t total = 0;
  std::vector<int64_t> over;  // queries with more than kCap matches
  for (int64_t i = 0; i < q; ++i) {
    res->offsets[i] = total;
    total += hc[i];
    if (hc[i] > static_cast<uint64_t>(kCap)) over.push_back(i);
  }
  res->offsets[q] = total;
  res->idx.resize(total);
  if (want_dist) res->dist.resize(total);
  if (total == 0) return SC_OK;
  {
    DevBuf off, oi, od;
    SC_HIP(off.alloc(sizeof(uint64_t) * (q + 1), s));
    SC_HIP(hipMemcpyAsync(off.p, res->offsets.data(), sizeof(uint64_t) * (q + 1),
                          hipMemcpyHostToDevice, s));
    SC_HIP(oi.alloc(sizeof(int64_t) * total, s));
    if (want_dist) SC_HIP(od.alloc(sizeof(double) * total, s));
    constexpr int kWaves = 4;
    hipLaunchKernelGGL(radius_compact_kernel, dim3(static_cast<unsigned>((q + kWaves - 1) / kWaves)),
                       dim3(64 * kWaves), 0, s, ci.as<int64_t>(),
                       want_dist ? cd.as<double>() : nullptr, kCap, cnt.as<uint64_t>(),
                       off.as<uint64_t>(), q, oi.as<int64_t>(), want_dist ? od.as<double>() : nullptr);
    SC_HIP(hipGetLastError());
    if (int rc = download_staged(res->idx.data(), oi.p, sizeof(int64_t) * total, s)) return rc;
    if (want_dist)
      if (int rc = download_staged(res->dist.data(), od.p, sizeof(double) * total, s)) return rc;
  }
  if (!over.empty()) {
    const int64_t m = static_cast<int64_t>(over.size());
    sc_radius_result sub;
    if (int rc = search_subset<T, M>(ix, dq, over, p, radius, &sub, want_dist, s)) return rc;
    for (int64_t j = 0; j < m; ++j) {
      const int64_t i = over[j];
      const uint64_t b = sub.offsets[j], c = sub.offsets[j + 1] - b;
      if (c != hc[i]) return fail(SC_ERR_DEVICE, "radius search: a query's match count differs between passes");
      std::copy(sub.idx.begin() + b, sub.idx.begin() + b + c, res->idx.begin() + res->offsets[i]);
      if (want_dist)
        std::copy(sub.dist.begin() + b, sub.dist.begin() + b + c, res->dist.begin() + res->offsets[i]);
    }
  }
  SC_HIP(hipStreamSynchronize(s));
  return SC_OK;
}

template <typename T, int M>
int run_radius(const sc_index* ix, const T* dq, int64_t q, double p, double radius,
               sc_radius_result* res, bool want_dist, bool allow_cap, hipStream_t s) {
  const int64_t n = static_cast<int64_t>(ix->n);
  const int ld = static_cast<int>(ix->ld);
  const int64_t nqt = (q + QT - 1) / QT;
  const int64_t tiles = std::max<int64_t>(1, (n + RT - 1) / RT);
  int64_t nseg = std::min<int64_t>(std::max<int64_t>(1, (4096 + nqt - 1) / nqt), tiles);
  nseg = std::min<int64_t>(nseg, 65535);
  const int64_t seg_tiles = (tiles + nseg - 1) / nseg;
  nseg = (tiles + seg_tiles - 1) / seg_tiles;
  const int64_t seg_len = seg_tiles * RT;
  // Conservative bound on the sum for the exact test d <= radius.
  double bound;
  if (M == kEuclid)
    bound = radius * radius * (1.0 + 1e-12) + 1e-300;
  else if (M == kManhattan)
    bound = radius;
  else
    bound = std::pow(radius, p) * (1.0 + 1e-9) + 1e-300;
  if (!std::isfinite(bound)) bound = INFINITY;
  // (a larger bound would admit sums that overflow in the rows' type)
  if constexpr (M == kEuclid) {
    if (allow_cap && bound < sum_limit<T>() &&
        static_cast<double>(q) * static_cast<double>(n) > kSweepMinPairs) {
      if (q <= kSweepQueries) {
        const int rc = run_radius_f64<T>(ix, dq, q, radius, bound, res, want_dist, s);
        if (rc != SC_ERR_OUT_OF_MEMORY) return rc;
        clear_error();  // the two passes keep nothing beside the rows
        return run_radius<T, M>(ix, dq, q, p, radius, res, want_dist, false, s);
      }
      res->q = static_cast<size_t>(q);
      res->offsets.assign(1, 0);
      for (int64_t b0 = 0; b0 < q; b0 += kSweepQueries) {
        sc_radius_result part;
        if (int rc = run_radius<T, M>(ix, dq + b0 * ld, std::min(kSweepQueries, q - b0), p, radius, &part,
                                      want_dist, true, s))
          return rc;
        const uint64_t base = res->offsets.back();
        for (size_t i = 1; i < part.offsets.size(); ++i) res->offsets.push_back(base + part.offsets[i]);
        res->idx.insert(res->idx.end(), part.idx.begin(), part.idx.end());
        res->dist.insert(res->dist.end(), part.dist.begin(), part.dist.end());
      }
      return SC_OK;
    }
  }
  if (allow_cap && nseg == 1 &&
      static_cast<double>(q) * static_cast<double>(kCap) * (want_dist ? 16.0 : 8.0) <= kCapBytes)
    return run_radius_capped<T, M>(ix, dq, q, p, radius, bound, res, want_dist, s);

  DevBuf cnt;
  SC_HIP(cnt.alloc(sizeof(uint64_t) * q * nseg, s));
  dim3 grid(static_cast<unsigned>(nqt), static_cast<unsigned>(nseg));
  hipLaunchKernelGGL((radius_kernel<T, M, kCount, false>), grid, dim3(NT), 0, s, static_cast<const T*>(ix->rows),
                     n, ld, static_cast<int>(ix->d), dq, q, p, radius, bound, seg_len, static_cast<int>(nseg),
                     cnt.as<uint64_t>(), nullptr, nullptr, int64_t{0});
  SC_HIP(hipGetLastError());
  std::vector<uint64_t> hc(static_cast<size_t>(q * nseg));
  SC_HIP(hipMemcpyAsync(hc.data(), cnt.p, sizeof(uint64_t) * hc.size(), hipMemcpyDeviceToHost, s));
  SC_HIP(hipStreamSynchronize(s));
  // exclusive scan in (query, segment) order = CSR offsets in index order
  res->q = static_cast<size_t>(q);
  res->offsets.assign(static_cast<size_t>(q) + 1, 0);
  uint64_t total = 0;
  for (int64_t i = 0; i < q; ++i) {
    res->offsets[i] = total;
    for (int64_t sg = 0; sg < nseg; ++sg) {
      const uint64_t c = hc[i * nseg + sg];
      hc[i * nseg + sg] = total;
      total += c;
    }
  }
  res->offsets[q] = total;
  res->idx.resize(total);
  if (want_dist) res->dist.resize(total);
  if (total == 0) return SC_OK;
  DevBuf oi, od;
  SC_HIP(oi.alloc(sizeof(int64_t) * total, s));
  if (want_dist) SC_HIP(od.alloc(sizeof(double) * total, s));
  SC_HIP(hipMemcpyAsync(cnt.p, hc.data(), sizeof(uint64_t) * hc.size(), hipMemcpyHostToDevice, s));
  if (want_dist)
    hipLaunchKernelGGL((radius_kernel<T, M, kFill, true>), grid, dim3(NT), 0, s,
                       static_cast<const T*>(ix->rows), n, ld, static_cast<int>(ix->d), dq, q, p,
                       radius, bound, seg_len, static_cast<int>(nseg), cnt.as<uint64_t>(),
                       oi.as<int64_t>(), od.as<double>(), int64_t{0});
  else
    hipLaunchKernelGGL((radius_kernel<T, M, kFill, false>), grid, dim3(NT), 0, s,
                       static_cast<const T*>(ix->rows), n, ld, static_cast<int>(ix->d), dq, q, p,
                       radius, bound, seg_len, static_cast<int>(nseg), cnt.as<uint64_t>(),
                       oi.as<int64_t>(), nullptr, int64_t{0});
  SC_HIP(hipGetLastError());
  // staged through the pinned buffers (parallel host copies)
  if (int rc = download_staged(res->idx.data(), oi.p, sizeof(int64_t) * total, s)) return rc;
  if (want_dist)
    if (int rc = download_staged(res->dist.data(), od.p, sizeof(double) * total, s)) return rc;
  SC_HIP(hipStreamSynchronize(s));
  return SC_OK;
}

template <typename T>
int radius_dispatch(const sc_index* ix, const void* dq, int64_t q, sc_metric metric, int p,
                    double radius, sc_radius_result* res, bool want_dist, hipStream_t s) {
  const T* qs = static_cast<const T*>(dq);
  switch (metric) {
    case SC_EUCLIDIAN:
      return run_radius<T, kEuclid>(ix, qs, q, 2.0, radius, res, want_dist, true, s);
    case SC_MANHATTAN:
      return run_radius<T, kManhattan>(ix, qs, q, 1.0, radius, res, want_dist, true, s);
    case SC_MINKOWSKI:
      return run_radius<T, kMinkowski>(ix, qs, q, static_cast<double>(p), radius, res, want_dist,
                                         true, s);
  }
  return fail(SC_ERR_UNSUPPORTED, "unknown metric");
}

}  // namespace

int radius_search_device(const sc_index* index, const void* d_queries, int64_t q,
                         sc_metric metric, int p, double radius, sc_radius_result* res,
                         hipStream_t s, bool want_dist) {
  res->q = static_cast<size_t>(q);
  res->offsets.assign(static_cast<size_t>(q) + 1, 0);
  res->idx.clear();
  res->dist.clear();
  if (q == 0 || index->n == 0) return SC_OK;
  return index->dtype == SC_F64
             ? radius_dispatch<double>(index, d_queries, q, metric, p, radius, res, want_dist, s)
             : radius_dispatch<float>(index, d_queries, q, metric, p, radius, res, want_dist, s);
}

}  // namespace sc

using namespace sc;

extern "C" {

int sc_radius_search(const sc_index* index, const void* queries, size_t q, double radius,
                     sc_metric metric, uint16_t p, sc_radius_result** out) {
  clear_error();
  if (!index || !out) return fail(SC_PARAMETERS_ERROR, "null argument");
  *out = nullptr;
  // linear_search.rs:90-95
  if (!(radius > 0.0)) return fail(SC_FIND_FAILED, "radius should be > 0");
  if (metric != SC_EUCLIDIAN && metric != SC_MANHATTAN && metric != SC_MINKOWSKI)
    return fail(SC_ERR_UNSUPPORTED, "unknown metric");
  if (metric == SC_MINKOWSKI && p < 1) return fail(SC_ERR_PANIC, "p must be at least 1");
  auto* res = new sc_radius_result();
  res->q = q;
  res->offsets.assign(q + 1, 0);
  if (q == 0 || index->n == 0) {
    *out = res;
    return SC_OK;
  }
  if (!queries) {
    delete res;
    return fail(SC_PARAMETERS_ERROR, "null queries");
  }
  hipError_t e = hipSetDevice(index->device);
  if (e != hipSuccess) {
    delete res;
    return hip_fail(e, "hipSetDevice");
  }
  hipStream_t s = stream_for(index);
  int rc;
  {
    DevBuf dq;
    e = dq.alloc(q * index->ld * elem_size(index->dtype), s);
    if (e != hipSuccess) {
      delete res;
      return hip_fail(e, "alloc queries");
    }
    rc = upload_padded(queries, index->dtype, q, index->d, index->ld, dq.p, s);
    if (rc == SC_OK)
      rc = radius_search_device(index, dq.p, static_cast<int64_t>(q), metric, p, radius, res, s);
  }
  if (rc != SC_OK) {
    delete res;
    return rc;
  }
  *out = res;
  return SC_OK;
}

size_t sc_radius_result_total(const sc_radius_result* r) { return r ? r->idx.size() : 0; }

int sc_radius_result_copy(const sc_radius_result* r, uint64_t* offsets, int64_t* idx,
                          double* dist) {
  clear_error();
  if (!r) return fail(SC_PARAMETERS_ERROR, "null result");
  if (offsets) std::copy(r->offsets.begin(), r->offsets.end(), offsets);
  if (idx) std::copy(r->idx.begin(), r->idx.end(), idx);
  if (dist) std::copy(r->dist.begin(), r->dist.end(), dist);
  return SC_OK;
}

void sc_radius_result_free(sc_radius_result* r) { delete r; }

}  // extern "C"
