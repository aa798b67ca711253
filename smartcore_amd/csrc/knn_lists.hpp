// What the candidate-list forms of the exact kNN search share: the levels of
// a scan, the candidate lists, the selection of thresholds, and the final
// rescoring and heap replay (LinearKNNSearch::find, linear_search.rs:52-84).
//
// A form scans the index in a dense prefix and levels whose row ranges grow
// geometrically; a level's candidates are the rows whose lower bound is below
// the k-th smallest upper bound of all earlier candidates, so the lists are a
// superset of the rows that enter the reference heap, in row order.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "common.hpp"
#include "heap.hpp"
#include "metric.hpp"

namespace sc {
namespace {

constexpr int64_t kDenseRows = 1024;
constexpr int kListTile = 128;       // rows per tile of every scan
// The finish's threads per query: with a workgroup of 128 for each query, the
// 256 CUs are busy from 512 queries on; fewer get more threads each.
constexpr int kFinishThreads = 128;
constexpr int kFinishWide = 512;
constexpr int64_t kFinishWideQueries = 512;
constexpr size_t kFinishWideLds = 8192;  // beside 52 KB of tiles and batch
// candidates rescored and replayed at a time
constexpr int finish_batch(int threads) { return threads == kFinishWide ? 1024 : 512; }
constexpr int kSelectWaves = 4;
constexpr int kMaxLevels = 8;

__global__ void zero_words_kernel(uint32_t* p, int64_t n) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x)
    p[i] = 0u;
}

// The k smallest values a wavefront has seen, ascending in lanes 0 .. k-1.
template <typename V>
__device__ __forceinline__ V none_seen();
// "none seen".  The compiler keeps a uniform f64 in a scalar register pair
// and writes the constant +inf there with one s_mov_b64, whose literal holds
// the low half only (it reads back as 0.0); the empty asm keeps the value in
// vector registers.
template <>
__device__ __forceinline__ double none_seen<double>() {
  double inf = INFINITY;
  asm volatile("" : "+v"(inf));
  return inf;
}
template <>
__device__ __forceinline__ uint32_t none_seen<uint32_t>() {
  return 0xffffffffu;
}
template <typename V>
struct KSmallest {
  V b;    // lane's entry
  V kth;
  __device__ __forceinline__ void clear() { b = kth = none_seen<V>(); }
  __device__ __forceinline__ void insert(V x, int lane, int k) {
    const V prev = __shfl_up(b, 1);
    if (lane < k && x < b) b = (lane > 0 && x < prev) ? prev : x;
    kth = lane_value(b, k - 1);
  }
  // one value per lane
  __device__ __forceinline__ void take_lanes(V x, int lane, int k) {
    uint64_t m = __ballot(x < kth);
    while (m) {
      insert(lane_value(x, __builtin_ctzll(m)), lane, k);
      m &= m - 1;
      m &= __ballot(x < kth);
    }
  }
  // the entries of src[0 .. n)
  __device__ __forceinline__ void take(const V* src, uint32_t n, int lane, int k) {
    for (uint32_t c0 = 0; c0 < n; c0 += 64)
      take_lanes(c0 + lane < n ? src[c0 + lane] : none_seen<V>(), lane, k);
  }
};

// One level of the scan.  Its (query tile, row tile) pairs, query tiles
// outermost, are dealt to the workgroups in contiguous runs of `per`, so all
// end together; the part of a run inside one query tile is a piece, with one
// candidate list per query.  The pieces of query tile qt are the workgroups
// from qt * tiles / per on.
struct Level {
  int64_t row0, tiles, per, groups;
  int lists;  // per query
  int cap;    // entries per list
  int64_t entry0, list0;  // where the level's lists begin (per query)
};
template <typename V>
struct ScanOut {
  uint32_t* idx;    // q x entries
  V* u;             // q x entries: an upper bound of each
  uint32_t* count;  // q x lists
  int64_t entries, lists;  // per query, all levels
};

// The k smallest upper bounds of the earlier levels (seed) and the entries
// of one level's lists, in place.
template <typename V>
__global__ __launch_bounds__(64 * kSelectWaves) void select_level_kernel(Level lv, ScanOut<V> in,
                                                                         int64_t q, int k,
                                                                         V* __restrict__ seed) {
  const int lane = threadIdx.x & 63;
  const int64_t qi = static_cast<int64_t>(blockIdx.x) * kSelectWaves + (threadIdx.x >> 6);
  if (qi >= q) return;  // the whole wave
  KSmallest<V> ks;
  ks.b = lane < k ? seed[qi * k + lane] : none_seen<V>();
  ks.kth = lane_value(ks.b, k - 1);
  const uint32_t* cc = in.count + qi * in.lists + lv.list0;
  const V* u = in.u + qi * in.entries + lv.entry0;
  // 64 lists at a time, lane = list: entry r of all of them in one load (the
  // lists are short; their order does not matter here)
  for (int l0 = 0; l0 < lv.lists; l0 += 64) {
    const uint32_t c = l0 + lane < lv.lists ? min(cc[l0 + lane], static_cast<uint32_t>(lv.cap)) : 0u;
    const V* ul = u + static_cast<int64_t>(l0 + lane) * lv.cap;
    for (uint32_t r = 0; __ballot(r < c) != 0; ++r) {
      const V x = r < c ? ul[r] : none_seen<V>();
      ks.take_lanes(x, lane, k);
    }
  }
  if (lane < k) seed[qi * k + lane] = ks.b;
}

// Where the lists of a query lie: list 0 is the dense prefix's (its own
// array), then each level's.
template <typename V>
struct Lists {
  const uint32_t* pre_idx;
  const uint32_t* pre_count;
  int pre_cap;
  ScanOut<V> out;
  int nlevels;
  Level lv[kMaxLevels];
};

// Whether a query row is staged in LDS (up to 32 KB of it).
template <typename T>
__host__ __device__ inline bool finish_staged(int ld) {
  return ld * sizeof(T) <= 32768;
}
template <typename T>
inline size_t finish_lds(int ld, int64_t lists) {
  return (finish_staged<T>(ld) ? sizeof(T) * ld : 0) + sizeof(uint32_t) * (lists + 2);
}

// S of every candidate and the heap replay (see the file comment).  The
// candidates are numbered across the lists by a prefix sum of the counts and
// taken a batch at a time: all threads compute their S, then the first
// wavefront replays the batch from LDS, 64 entries at a time.
template <typename T, int M, typename V, int THREADS>
__global__ __launch_bounds__(THREADS) void finish_kernel(
    const T* __restrict__ rows, int ld, const T* __restrict__ queries, int64_t q, int k, Lists<V> ls,
    int64_t* __restrict__ out_idx, double* __restrict__ out_dist, uint32_t* __restrict__ out_count,
    uint32_t* __restrict__ list, uint32_t* __restrict__ list_n,
    unsigned long long* __restrict__ total_cand) {
  constexpr int kBatch = finish_batch(THREADS);
  // the query row (unless it is too wide), then the lists' starts (nl + 1)
  extern __shared__ __align__(16) unsigned char finish_smem[];
  const bool staged = finish_staged<T>(ld);
  T* qrow = reinterpret_cast<T*>(finish_smem);
  uint32_t* start = reinterpret_cast<uint32_t*>(qrow + (staged ? ld : 0));
  __shared__ double s_S[kBatch];
  __shared__ uint32_t s_row[kBatch];
  __shared__ __align__(16) unsigned char tiles[THREADS / 64][kSumTileBytes];
  __shared__ uint32_t s_over;
  const int64_t qi = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int nl = 1 + static_cast<int>(ls.out.lists);
  if (tid == 0) s_over = 0u;
  if (staged)
    for (int j = tid; j < ld; j += THREADS) qrow[j] = queries[qi * ld + j];
  __syncthreads();
  // exclusive prefix sum of the counts: each thread takes a run of lists
  __shared__ uint32_t s_wave[THREADS / 64];
  const int run = (nl + THREADS - 1) / THREADS;
  const int l0 = min(tid * run, nl), l1 = min(l0 + run, nl);
  uint32_t sum = 0;
  bool over = false;
  for (int l = l0; l < l1; ++l) {
    uint32_t c;
    int cap = ls.pre_cap;
    if (l == 0) {
      c = ls.pre_count[qi];
    } else {
      c = ls.out.count[qi * ls.out.lists + l - 1];
      cap = ls.lv[0].cap;
      for (int v = 1; v < ls.nlevels; ++v)
        if (l - 1 >= ls.lv[v].list0) cap = ls.lv[v].cap;
    }
    over = over || c > static_cast<uint32_t>(cap);
    start[l] = c;
    sum += c;
  }
  uint32_t inc = sum;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t up = __shfl_up(inc, o);
    if (lane >= o) inc += up;
  }
  if (lane == 63) s_wave[tid >> 6] = inc;
  if (over) s_over = 1u;
  __syncthreads();
  uint32_t at = inc - sum;
  for (int w = 0; w < (tid >> 6); ++w) at += s_wave[w];
  for (int l = l0; l < l1; ++l) {
    const uint32_t c = start[l];
    start[l] = at;
    at += c;
  }
  if (tid == THREADS - 1) start[nl] = at;
  if (tid == 0 && s_over) {
    list[atomicAdd(list_n, 1u)] = static_cast<uint32_t>(qi);
    out_count[qi] = 0u;
  }
  __syncthreads();
  if (s_over) return;
  const uint32_t total = start[nl];
  double hd = INFINITY, top = INFINITY;
  uint32_t hi = 0xffffffffu;
  for (uint32_t e0 = 0; e0 < total; e0 += kBatch) {
    const uint32_t m = min(total - e0, static_cast<uint32_t>(kBatch));
    for (uint32_t b0 = tid & ~63u; b0 < m; b0 += THREADS) {  // a wavefront's 64
      const uint32_t e = min(b0 + lane, m - 1);
      // the list of candidate e0 + e: the last whose start is at or below it
      int lo = 0, hi_l = nl;
      while (hi_l - lo > 1) {
        const int mid = (lo + hi_l) >> 1;
        if (start[mid] <= e0 + e)
          lo = mid;
        else
          hi_l = mid;
      }
      const uint32_t at = e0 + e - start[lo];
      uint32_t row;
      if (lo == 0) {
        row = ls.pre_idx[qi * ls.pre_cap + at];
      } else {
        int v = 0;
        while (v + 1 < ls.nlevels && lo - 1 >= ls.lv[v + 1].list0) ++v;
        row = ls.out.idx[qi * ls.out.entries + ls.lv[v].entry0 +
                         (lo - 1 - ls.lv[v].list0) * ls.lv[v].cap + at];
      }
      const double s = staged ? wave_exact_sums<T, M>(qrow, rows, row, ld, tiles[tid >> 6])
                              : exact_sum<T, M>(queries + qi * ld, rows + static_cast<int64_t>(row) * ld, ld);
      if (b0 + lane < m) {
        s_S[e] = s;
        s_row[e] = row;
      }
    }
    __syncthreads();
    if (tid < 64) {
      for (uint32_t c0 = 0; c0 < m; c0 += 64) {
        const bool valid = c0 + lane < m;
        const double dv = valid ? finalize<M>(s_S[c0 + lane], 1.0) : 0.0;
        const uint32_t row = valid ? s_row[c0 + lane] : 0u;
        uint64_t b = __ballot(valid && dv < top);
        while (b) {
          const int src = __builtin_ctzll(b);
          lane_heap_push_root(hd, hi, lane, k, lane_value(dv, src),
                              static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(row), src)));
          top = lane_value(hd, 0);
          b &= b - 1;
          b &= __ballot(valid && dv < top);
        }
      }
    }
    __syncthreads();
  }
  if (tid < 64) {
    // (only when asked for: one address for all queries)
    if (total_cand && lane == 0) atomicAdd(total_cand, static_cast<unsigned long long>(total));
    lane_heap_store(hd, hi, lane, k, out_idx + qi * k, out_dist + qi * k, out_count + qi);
  }
}

// 20 queries over 600,000 x 32 f32 rows sorted by class, whose first rows tell
// little of the others (tens of thousands of candidates each), Manhattan:
// 2.8 ms with 128 threads per query, 1.1 with 512; one query with the usual few
// hundred: 45 and 37 us.
template <typename T, int M, typename V>
void launch_finish(const T* rows, int ld, const T* queries, int64_t q, int k, const Lists<V>& ls,
                   int64_t* out_idx, double* out_dist, uint32_t* out_count, uint32_t* list,
                   uint32_t* list_n, unsigned long long* total_cand, hipStream_t s) {
  const size_t lds = finish_lds<T>(ld, ls.out.lists);
  const dim3 grid(static_cast<unsigned>(q));
  if (q <= kFinishWideQueries && lds <= kFinishWideLds)
    hipLaunchKernelGGL((finish_kernel<T, M, V, kFinishWide>), grid, dim3(kFinishWide), lds, s, rows, ld,
                       queries, q, k, ls, out_idx, out_dist, out_count, list, list_n, total_cand);
  else
    hipLaunchKernelGGL((finish_kernel<T, M, V, kFinishThreads>), grid, dim3(kFinishThreads), lds, s, rows, ld,
                       queries, q, k, ls, out_idx, out_dist, out_count, list, list_n, total_cand);
}

// The rows at which the levels begin and end: the dense prefix of `cols`
// rows, then m ranges growing by the same factor (at most 16: a level leaves
// k (factor - 1) candidates per query, one more costs a scan and a selection
// launch).
inline std::vector<int64_t> level_edges(int64_t n, int64_t cols) {
  std::vector<int64_t> edge{cols};
  if (n > cols) {
    const double span = static_cast<double>(n) / static_cast<double>(cols);
    const int m = std::max(1, std::min(kMaxLevels, static_cast<int>(std::ceil(std::log(span) / std::log(16.0)))));
    for (int i = 1; i < m; ++i)
      edge.push_back(std::max<int64_t>(
          edge.back() + kListTile,
          static_cast<int64_t>(cols * std::pow(span, double(i) / m)) / kListTile * kListTile));
    edge.push_back(n);
  }
  return edge;
}
// Expected running-k-th improvements over len rows in random order.
inline double expected_entrants(int k, double len) {
  return k * (1.0 + std::log(std::max(1.0, len / k)));
}
// Levels for qn queries in tiles of tile_q, dealt to about `groups` equal
// pieces.
template <typename V>
inline void plan_levels(const std::vector<int64_t>& edge, int64_t qn, int tile_q, int64_t groups, int k,
                        Level (&lv)[kMaxLevels], ScanOut<V>& o) {
  const int64_t nqt = (qn + tile_q - 1) / tile_q;
  o.entries = o.lists = 0;
  for (size_t i = 0; i + 1 < edge.size(); ++i) {
    Level& v = lv[i];
    v.row0 = edge[i];
    v.tiles = (edge[i + 1] - edge[i] + kListTile - 1) / kListTile;
    const int64_t items = nqt * v.tiles;
    v.per = std::max<int64_t>(1, (items + groups - 1) / groups);
    v.groups = (items + v.per - 1) / v.per;
    v.lists = static_cast<int>(std::min<int64_t>((v.tiles + v.per - 1) / v.per + 1, v.tiles));
    const int64_t len = std::min<int64_t>(v.per * kListTile, v.tiles * kListTile);
    // a tile that passes whole, one look's growth, and the running-k-th
    // improvements after it with room to spare
    v.cap = static_cast<int>(std::min<int64_t>(
        len, kListTile + std::max(2 * k, 32) +
                 static_cast<int64_t>(4.0 * expected_entrants(k, static_cast<double>(len)))));
    v.entry0 = o.entries;
    v.list0 = o.lists;
    o.entries += static_cast<int64_t>(v.lists) * v.cap;
    o.lists += v.lists;
  }
}

// The candidate store of a call is bounded by batches of queries, whole query
// tiles of kListTile each.  A smaller batch has longer lists per query, so the
// size is found by halving; bytes(o) is what one query takes under plan o.  The
// last batch may be short and its queries then spread over more pieces (132,178
// queries, 300,000 rows, k = 10: 12 % more entries in all than the batches
// before it), so the store is the larger of the two.
struct Batches {
  int64_t queries;         // of every batch but a short last one
  int64_t entries, lists;  // of the store, all queries of a batch
};
template <typename V, typename Plan, typename Bytes>
inline Batches plan_batches(int64_t q, Plan plan, Bytes bytes, Level (&lv)[kMaxLevels], ScanOut<V>& o) {
  int64_t qb = q;
  for (;;) {
    plan(qb, lv, o);
    if (static_cast<double>(qb) * bytes(o) <= 1.5 * 1024.0 * 1024.0 * 1024.0 || qb <= kListTile) break;
    qb = std::max<int64_t>(kListTile, (qb / 2 + kListTile - 1) / kListTile * kListTile);
  }
  Batches b{qb, o.entries * qb, o.lists * qb};
  if (const int64_t last = q % qb; last != 0) {
    Level llv[kMaxLevels];
    ScanOut<V> lo{};
    plan(last, llv, lo);
    b.entries = std::max(b.entries, lo.entries * last);
    b.lists = std::max(b.lists, lo.lists * last);
  }
  return b;
}

}  // namespace
}  // namespace sc
