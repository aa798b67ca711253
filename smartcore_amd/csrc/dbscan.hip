// DBSCAN::fit and DBSCAN::predict (cluster/dbscan.rs:274-397) over a device
// index.
//
// The distance work -- find_radius (linear_search.rs:89-108) of every row,
// O(n^2 d) -- runs on the device: for Euclidian as a sweep of row pairs (see
// "Euclidian fit"), for the other metrics as one batched radius search (each
// row's neighbours in index order, which is exactly the list find_radius
// returns).
//
// The reference's expansion loop (outer loop over the rows, `neighbors`
// used as a stack) gives these labels, which are computed here without the
// loop's order:
//   - core rows (at least min_samples neighbours, the row itself included)
//     joined by neighbour edges form the clusters, and the outer loop starts
//     each at its smallest core row, so cluster k is the component whose
//     smallest core row is the k-th such row in index order;
//   - every other row takes the first cluster whose expansion reaches it,
//     i.e. the lowest-numbered cluster among its core neighbours (clusters
//     are expanded one at a time, in order), or -1 when it has none.
// The components come from a union-find on the device over the core rows'
// edges (links always point a root at a smaller root, so a component's root
// is its smallest row); with neighbour lists the numbering and the non-core
// rows (whose lists are shorter than min_samples) are done on the host.  predict searches its
// queries the same way and takes the first most frequent label (which_max,
// tree/decision_tree_classifier.rs:490-502).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "common.hpp"
#include "metric.hpp"
#include "mfma64.hpp"

using namespace sc;

namespace {

// Union-find in one array, the larger of two trees' rows always under the
// smaller, so that a tree's root is its smallest row.
//
// Every value ever stored in parent[x] is an ancestor of x and at most x.  A
// read may be stale (another die's cache): it then gives an earlier, that is a
// lower, ancestor, and what it takes for a root is set right by the swap, which
// is not stale.  Pointing a row at its grandparent on the way (path splitting)
// needs no swap: the row has a parent by then, and only roots are linked.
__device__ uint32_t dbscan_rep(uint32_t* parent, uint32_t x) {
  for (;;) {
    const uint32_t up = parent[x];
    if (up == x) return x;
    const uint32_t above = parent[up];
    if (above == up) return up;
    parent[x] = above;
    x = above;
  }
}

// Joins the trees of u and v: Rem's algorithm (Dijkstra, 1976) without its
// splicing.  Of the two rows, the one with the larger parent goes up; where it
// has come to a root, that is linked under the other's parent by a
// compare-and-swap.  The larger parent falls with every round, and the walk ends
// where the two paths meet, which need not be at the root.
__device__ void dbscan_link(uint32_t* parent, uint32_t u, uint32_t v) {
  uint32_t pu = parent[u], pv = parent[v];
  while (pu != pv) {
    if (pu < pv) {
      const uint32_t x = u, px = pu;
      u = v;
      pu = pv;
      v = x;
      pv = px;
    }
    if (pu == u) {
      pu = atomicCAS(&parent[u], u, pv);
      if (pu == u) return;
    } else {
      const uint32_t above = parent[pu];
      if (above != pu) parent[u] = above;
      u = pu;
      pu = above;
    }
  }
}

__global__ void dbscan_init_kernel(const uint64_t* __restrict__ off, int64_t n,
                                   uint64_t min_samples, uint8_t* __restrict__ core,
                                   uint32_t* __restrict__ parent) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    core[i] = off[i + 1] - off[i] >= min_samples ? 1 : 0;
    parent[i] = static_cast<uint32_t>(i);
  }
}

// One wavefront per row: a core row is joined with its core neighbours of
// smaller index (the relation is symmetric, so each edge is taken once).
__global__ void dbscan_union_kernel(const uint64_t* __restrict__ off,
                                    const int64_t* __restrict__ idx, int64_t n,
                                    const uint8_t* __restrict__ core, uint32_t* parent) {
  const int lane = threadIdx.x & 63;
  const int64_t waves = (static_cast<int64_t>(gridDim.x) * blockDim.x) >> 6;
  for (int64_t i = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) >> 6; i < n;
       i += waves) {
    if (!core[i]) continue;
    const uint64_t e1 = off[i + 1];
    for (uint64_t e = off[i] + lane; e < e1; e += 64) {
      const int64_t j = idx[e];
      if (j < i && core[j]) dbscan_link(parent, static_cast<uint32_t>(i), static_cast<uint32_t>(j));
    }
  }
}

// The component root of every core row (0xffffffff for the others).
__global__ void dbscan_root_kernel(int64_t n, const uint8_t* __restrict__ core, uint32_t* parent,
                                   uint32_t* __restrict__ root) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x)
    root[i] = core[i] ? dbscan_rep(parent, static_cast<uint32_t>(i)) : 0xffffffffu;
}

// ---- Euclidian fit without neighbour lists ----
//
// Distances are symmetric bit for bit (a - b and b - a square alike), so the
// pairs below the diagonal are enough: one triangular sweep of 128 x 128
// FP64 MFMA tiles (mfma64.hpp) writes the (row, smaller row) pairs whose
// bound passes the radius, in no order; `verify` decides each with the
// reference's sum and counts both ends' neighbours; `join` joins the core
// rows of the remaining pairs; clusters are numbered by their smallest core
// row with a prefix sum, and a pair with one core end offers its cluster to
// the other.  Nothing but the labels goes to the host.
//
// The sweep does n^2 / 2 distances whatever the radius, so from kGroupMinRows
// rows on the rows are first put in an order of their own: each goes to the
// nearest of up to 128 pivots (rows taken at even steps), the groups are laid
// one after another, each from a tile's edge, and every tile of 128 rows gets
// its bounding box.  A tile pair whose boxes are further apart than the
// radius (in the bound's terms, so no pair that the reference would count)
// is skipped.  Any order gives the same pairs, and so the same labels.  The
// grouping costs about 128 distances per row.  200,000 x 8 rows in ten
// clusters with 55 neighbours each: 11.2 ms without groups, 3.2 with them (the
// sweep 2.35); 91 when the neighbour lists went to the host.  Fewer rows are
// swept whole in the time the grouping takes (32,768 rows of that kind: 0.44
// ms with groups and 0.47 without; 16,384: 0.42 and 0.24).
constexpr int64_t kGroupMinRows = 32768;
constexpr int kMaxPivots = 128;
constexpr int kPivotDims = 64;  // values of a row that the grouping looks at, at most
constexpr int kPivotStep = 16;  // pivots per pass over a row's values
constexpr uint32_t kNoRow = 0xffffffffu;

// One group per 512 rows: half a tile of padding each is an eighth.
int pivot_count(int64_t n) {
  return static_cast<int>(std::min<int64_t>(kMaxPivots, n / 512 / kPivotStep * kPivotStep));
}

// pivots[j * P + p]: value j of pivot p.
template <typename T>
__global__ void dbscan_pivots_kernel(const T* __restrict__ rows, int64_t n, int ld, int dims, int P,
                                     double* __restrict__ pivots) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= P * dims) return;
  const int j = e / P, p = e % P;
  pivots[e] = static_cast<double>(rows[static_cast<int64_t>(p) * n / P * ld + j]);
}

// Group of every row (P: the rows that are left out) and the groups' sizes.
// The pivots' values are the same for all lanes and come through the scalar
// cache, kPivotStep per load.
template <typename T>
__global__ __launch_bounds__(256) void dbscan_group_kernel(const T* __restrict__ rows, int64_t n,
                                                           int ld, int dims, int P,
                                                           const double* __restrict__ pivots,
                                                           const double* __restrict__ y2m,
                                                           uint8_t* __restrict__ group,
                                                           uint32_t* __restrict__ sizes) {
  __shared__ uint32_t h[kMaxPivots + 1];
  for (int g = threadIdx.x; g <= P; g += 256) h[g] = 0;
  __syncthreads();
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i < n) {
    const T* x = rows + i * ld;
    int which = 0;
    double best = INFINITY;
    for (int p0 = 0; p0 < P; p0 += kPivotStep) {
      double acc[kPivotStep];
#pragma unroll
      for (int u = 0; u < kPivotStep; ++u) acc[u] = 0.0;
#pragma unroll 2
      for (int j = 0; j < dims; ++j) {
        const double xj = static_cast<double>(x[j]);
        const double* pv = pivots + j * P + p0;
#pragma unroll
        for (int u = 0; u < kPivotStep; ++u) {
          const double df = xj - pv[u];
          acc[u] = __builtin_fma(df, df, acc[u]);
        }
      }
#pragma unroll
      for (int u = 0; u < kPivotStep; ++u)
        if (acc[u] < best) {
          best = acc[u];
          which = p0 + u;
        }
    }
    if (y2m[i] == INFINITY) which = P;
    group[i] = static_cast<uint8_t>(which);
    atomicAdd(&h[which], 1u);
  }
  __syncthreads();
  for (int g = threadIdx.x; g <= P; g += 256)
    if (h[g]) atomicAdd(&sizes[g], h[g]);
}

// The row of every place: groups one after another, each from a multiple of
// kMR (places between them keep kNoRow); the order inside a group is free.
constexpr int kPlaceThreads = 1024;
__global__ __launch_bounds__(kPlaceThreads) void dbscan_place_kernel(
    int64_t n, int P, const uint8_t* __restrict__ group, const uint32_t* __restrict__ sizes,
    uint32_t* __restrict__ taken, uint32_t* __restrict__ place) {
  __shared__ uint32_t padded[kMaxPivots + 1], h[kMaxPivots + 1], at[kMaxPivots + 1];
  const int tid = threadIdx.x;
  if (tid <= P) {
    padded[tid] = (sizes[tid] + kMR - 1) / kMR * kMR;
    h[tid] = 0;
  }
  __syncthreads();
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kPlaceThreads + tid;
  const int g = i < n ? group[i] : 0;
  const uint32_t rank = i < n ? atomicAdd(&h[g], 1u) : 0u;
  __syncthreads();
  if (tid <= P && h[tid]) {
    uint32_t a = 0;
    for (int u = 0; u < tid; ++u) a += padded[u];
    at[tid] = a + atomicAdd(&taken[tid], h[tid]);
  }
  __syncthreads();
  if (i < n) place[at[g] + rank] = static_cast<uint32_t>(i);
}

__global__ void dbscan_empty_kernel(int64_t m, uint32_t* __restrict__ place) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < m;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x)
    place[i] = kNoRow;
}

// The rows and norms in their places (16 bytes per thread); empty places are
// zero rows that take no part.
template <typename T>
__global__ void dbscan_gather_kernel(const T* __restrict__ rows, const double* __restrict__ y2m,
                                     int64_t m, int ld, const uint32_t* __restrict__ place,
                                     T* __restrict__ grows, double* __restrict__ gy2m) {
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  const int pieces = ld * static_cast<int>(sizeof(T)) / 16;
  const int64_t total = m * pieces;
  for (int64_t e = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; e < total;
       e += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t t = e / pieces;
    const int c = static_cast<int>(e - t * pieces);
    const uint32_t r = place[t];
    u4 v = {0u, 0u, 0u, 0u};
    if (r != kNoRow) v = reinterpret_cast<const u4*>(rows + static_cast<int64_t>(r) * ld)[c];
    reinterpret_cast<u4*>(grows + t * ld)[c] = v;
    if (c == 0) gy2m[t] = r != kNoRow ? y2m[r] : INFINITY;
  }
}

// box[j * 2 nt + t], box[(2 j + 1) nt + t]: lowest and highest value j of the
// rows of tile t that take part (+inf, -inf: none).  A thread per (tile,
// value), neighbours reading one row.
template <typename T>
__global__ __launch_bounds__(256) void dbscan_boxes_kernel(const T* __restrict__ grows,
                                                           const double* __restrict__ gy2m, int64_t nt,
                                                           int ld, int d, double* __restrict__ box) {
  const int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t t = e / ld;
  const int j = static_cast<int>(e - t * ld);
  if (t >= nt || j >= d) return;
  const T* x = grows + t * kMR * ld + j;
  const double* y = gy2m + t * kMR;
  double lo = INFINITY, hi = -INFINITY;
  asm volatile("" : "+v"(lo), "+v"(hi));  // (a uniform 64-bit literal would lose its upper half)
#pragma unroll 16
  for (int r = 0; r < kMR; ++r) {
    const double v = static_cast<double>(x[static_cast<int64_t>(r) * ld]);
    const bool in = y[r] != INFINITY;
    lo = in && v < lo ? v : lo;
    hi = in && v > hi ? v : hi;
  }
  box[static_cast<int64_t>(2 * j) * nt + t] = lo;
  box[static_cast<int64_t>(2 * j + 1) * nt + t] = hi;
}

constexpr int kPairBuf = 112;  // pairs staged in LDS per wavefront (with the rest, half a CU's LDS)

__device__ __forceinline__ int64_t triangle_row(int64_t pos) {
  int64_t r = static_cast<int64_t>((sqrt(8.0 * static_cast<double>(pos) + 1.0) - 1.0) * 0.5);
  while (r * (r + 1) / 2 > pos) --r;
  while ((r + 1) * (r + 2) / 2 <= pos) ++r;
  return r;
}

// A sweep's pairs.  Each wavefront collects its own in an LDS buffer (a place
// is the buffer's fill plus the lane's rank in the hit mask) and empties it
// when the next mask may not fit, with one update of the global counter;
// pairs past cap are counted only.
struct PairSink {
  uint2* mine;
  uint32_t fill;  // the same in the whole wavefront
  uint2* pairs;
  unsigned long long cap;
  unsigned long long* cursor;
  __device__ __forceinline__ void flush(const MLane& ml) {
    unsigned long long base = 0;
    if (ml.lane == 0) base = atomicAdd(cursor, static_cast<unsigned long long>(fill));
    base = __shfl(base, 0);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    for (uint32_t e = ml.lane; e < fill; e += 64)
      if (base + e < cap) pairs[base + e] = mine[e];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    fill = 0;
  }
  // the hits of tile t of a sweep of query tile qt
  __device__ __forceinline__ void take(const MLane& ml, const MAcc& acc, const double (&th)[2],
                                       const double* y2, int64_t qt, int64_t t) {
    tile_hits(ml, acc, th, y2, [&](int, int j, int, int rl, bool hit, uint64_t m) {
      if (t == qt) {  // the diagonal tile: smaller rows only
        hit = hit && rl < ml.query_of(j);
        m = __ballot(hit);
      }
      const uint32_t c = static_cast<uint32_t>(__popcll(m));
      if (fill + c > kPairBuf) flush(ml);
      if (hit)
        mine[fill + __popcll(m & ml.below())] =
            make_uint2(static_cast<uint32_t>(qt * kMQ + ml.query_of(j)), static_cast<uint32_t>(t * kMR + rl));
      fill += c;
    });
  }
};

// The thresholds of a query tile.
__device__ __forceinline__ void pair_thresholds(const MLane& ml, const double* y2m, int64_t qt,
                                                Bound64 bd, double bound, double (&th)[2]) {
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const double x2 = y2m[qt * kMQ + ml.query_of(j)];
    // rows left out take no part; rows past the bound's range (NaN) pass
    // every test
    th[j] = x2 == INFINITY ? -INFINITY : acc_threshold(bd, bound, x2);
  }
}

// Every tile pair: tiles (qt, t <= qt) numbered qt (qt + 1) / 2 + t, dealt to
// the workgroups in contiguous runs.
template <typename T>
__global__ __launch_bounds__(kMT, 2) void dbscan_pairs_kernel(
    const T* __restrict__ rows, int64_t n, int ld, int d, const double* __restrict__ y2m, Bound64 bd,
    double bound, int64_t total, int64_t per, uint2* __restrict__ pairs, unsigned long long cap,
    unsigned long long* __restrict__ cursor) {
  __shared__ MSmem sm;
  __shared__ uint2 buf[kMT / 64][kPairBuf];
  const MLane ml;
  PairSink sink{buf[ml.wave], 0, pairs, cap, cursor};
  int64_t pos = static_cast<int64_t>(blockIdx.x) * per;
  const int64_t end = min(pos + per, total);
  while (pos < end) {
    const int64_t qt = triangle_row(pos);
    const int64_t tb = pos - qt * (qt + 1) / 2;
    const int64_t te = min(qt + 1, tb + (end - pos));
    double th[2];
    pair_thresholds(ml, y2m, qt, bd, bound, th);
    mfma64_sweep<T, false>(sm, rows, n, ld, d, y2m, rows, n, qt * kMQ, 0, tb, te,
                           [&](int64_t t, MAcc& acc, int par) { sink.take(ml, acc, th, sm.y2[par], qt, t); });
    pos += te - tb;
    __syncthreads();  // the sweep's LDS is staged anew
  }
  sink.flush(ml);
}

// The tile pairs whose boxes are within the radius.  An item is a query tile
// qt and a run of kRun tiles: the first threads test one tile's box each and
// the ones that remain are swept as one list.  Items are taken from a counter
// (the lists' lengths differ widely) until none is left.  swept: tile pairs taken.
constexpr int kRun = 128;
static_assert(kRun == 2 * 64 && kRun <= kMT, "two wavefronts test a run");
template <typename T>
__global__ __launch_bounds__(kMT, 2) void dbscan_near_pairs_kernel(
    const T* __restrict__ rows, int64_t nt, int ld, int d, const double* __restrict__ y2m,
    const double* __restrict__ box, Bound64 bd, double bound, double apart, int64_t items,
    uint2* __restrict__ pairs, unsigned long long cap, unsigned long long* __restrict__ cursor,
    unsigned long long* __restrict__ next, unsigned long long* __restrict__ swept) {
  __shared__ MSmem sm;
  __shared__ uint2 buf[kMT / 64][kPairBuf];
  __shared__ uint8_t list[kRun];
  __shared__ unsigned long long s_item;
  __shared__ uint32_t s_count[2];
  const MLane ml;
  const int tid = threadIdx.x;
  PairSink sink{buf[ml.wave], 0, pairs, cap, cursor};
  for (;;) {
    if (tid == 0) s_item = atomicAdd(next, 1ull);
    __syncthreads();
    const int64_t it = static_cast<int64_t>(s_item);
    if (it >= items) break;
    const int64_t qt = it % nt, t0 = it / nt * kRun;
    uint64_t near = 0;
    if (tid < kRun) {
      const int64_t t = t0 + tid;
      bool in = t <= qt;
      if (__ballot(in)) {
        const int64_t tc = min(t, nt - 1);
        double s = 0.0;
#pragma unroll 4
        for (int j = 0; j < d; ++j) {
          const double* lo = box + static_cast<int64_t>(2 * j) * nt;
          const double* hi = lo + nt;
          // (no rows: +inf apart)
          const double g = fmax(fmax(lo[qt] - hi[tc], lo[tc] - hi[qt]), 0.0);
          s = __builtin_fma(g, g, s);
        }
        in = in && !(s > apart);
      }
      near = __ballot(in);
      if (ml.lane == 0) s_count[ml.wave] = static_cast<uint32_t>(__popcll(near));
    }
    __syncthreads();
    const uint32_t count = s_count[0] + s_count[1];
    if (tid == 0 && count) atomicAdd(swept, static_cast<unsigned long long>(count));
    if ((near >> ml.lane) & 1)
      list[(ml.wave ? s_count[0] : 0u) + __popcll(near & ml.below())] = static_cast<uint8_t>(tid);
    __syncthreads();
    if (count == 0) continue;
    auto at = [&](int64_t e) { return t0 + __builtin_amdgcn_readfirstlane(static_cast<int>(list[e])); };
    double th[2];
    pair_thresholds(ml, y2m, qt, bd, bound, th);
    mfma64_sweep<T, false>(sm, rows, nt * kMR, ld, d, y2m, rows, nt * kMR, qt * kMQ, 0, 0, count,
                           [&](int64_t e, MAcc& acc, int par) { sink.take(ml, acc, th, sm.y2[par], qt, at(e)); },
                           at);
    __syncthreads();  // the sweep's LDS, the list and the item are written anew
  }
  sink.flush(ml);
}

// Decides each pair with the reference's distance: its ends' neighbour
// counts, or (no neighbours) an empty pair.  place: the rows that lie at the
// pair's places, which the pair holds from here on (null: the places are the
// rows).
template <typename T>
__global__ __launch_bounds__(256) void dbscan_verify_kernel(const T* __restrict__ rows, int ld,
                                                            double radius,
                                                            const uint32_t* __restrict__ place,
                                                            uint2* __restrict__ pairs,
                                                            unsigned long long cap,
                                                            const unsigned long long* __restrict__ cursor,
                                                            uint32_t* __restrict__ degree) {
  const unsigned long long m = min(*cursor, cap);
  for (unsigned long long e = static_cast<unsigned long long>(blockIdx.x) * blockDim.x + threadIdx.x;
       e < m; e += static_cast<unsigned long long>(gridDim.x) * blockDim.x) {
    uint2 p = pairs[e];
    const double s = exact_sum<T, kEuclid>(rows + static_cast<int64_t>(p.x) * ld, rows + static_cast<int64_t>(p.y) * ld, ld);
    if (__builtin_sqrt(s) <= radius) {
      if (place) {
        p = make_uint2(place[p.x], place[p.y]);
        pairs[e] = p;
      }
      atomicAdd(&degree[p.x], 1u);
      atomicAdd(&degree[p.y], 1u);
    } else {
      pairs[e].x = kNoRow;
    }
  }
}

// A row whose values are all finite is its own neighbour (distance 0).
__global__ void dbscan_self_kernel(const double* __restrict__ y2m, int64_t n,
                                   uint32_t* __restrict__ degree, uint32_t* __restrict__ parent) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    degree[i] = y2m[i] == INFINITY ? 0u : 1u;
    parent[i] = static_cast<uint32_t>(i);
  }
}

// Joins the core ends of every step-th pair.  Joining all pairs at once
// spends its time on walks and failed swaps at a few roots (0.45 ms for 5.5
// million pairs); a sixteenth of the pairs already joins nearly all of a
// cluster, and once every row points at its root the other pairs mostly find
// their ends joined with two loads (0.22 in all).
constexpr int kJoinSample = 16;
__global__ __launch_bounds__(256) void dbscan_join_kernel(const uint2* __restrict__ pairs,
                                                          unsigned long long cap,
                                                          const unsigned long long* __restrict__ cursor,
                                                          const uint32_t* __restrict__ degree,
                                                          uint64_t min_samples, int step,
                                                          uint32_t* parent) {
  const unsigned long long m = min(*cursor, cap);
  for (unsigned long long e = (static_cast<unsigned long long>(blockIdx.x) * blockDim.x + threadIdx.x) * step;
       e < m; e += static_cast<unsigned long long>(gridDim.x) * blockDim.x * step) {
    const uint2 p = pairs[e];
    if (p.x == kNoRow || degree[p.x] < min_samples || degree[p.y] < min_samples) continue;
    // (the same parent, whatever it is by now: the same tree)
    if (parent[p.x] != parent[p.y]) dbscan_link(parent, p.x, p.y);
  }
}

// Every row points at its root.
__global__ void dbscan_compress_kernel(int64_t n, uint32_t* parent) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x)
    parent[i] = dbscan_rep(parent, static_cast<uint32_t>(i));
}

// root[i] of every core row (0xffffffff for the others), and per block of
// kNumberBlock rows how many clusters start there (a core row that is its
// own root).
constexpr int kNumberBlock = 1024;
__global__ __launch_bounds__(kNumberBlock) void dbscan_roots_kernel(
    int64_t n, const uint32_t* __restrict__ degree, uint64_t min_samples, uint32_t* parent,
    uint32_t* __restrict__ root, uint32_t* __restrict__ starts) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kNumberBlock + threadIdx.x;
  uint32_t r = 0xffffffffu;
  if (i < n) {
    if (degree[i] >= min_samples) r = dbscan_rep(parent, static_cast<uint32_t>(i));
    root[i] = r;
  }
  const int c = __syncthreads_count(i < n && r == static_cast<uint32_t>(i));
  if (threadIdx.x == 0) starts[blockIdx.x] = static_cast<uint32_t>(c);
}

// Exclusive prefix sum of the block counts in place; the total after them.
__global__ __launch_bounds__(64) void dbscan_scan_kernel(uint32_t* __restrict__ starts, int64_t nb) {
  const int lane = threadIdx.x;
  uint32_t acc = 0;
  for (int64_t b0 = 0; b0 < nb; b0 += 64) {
    const uint32_t c = b0 + lane < nb ? starts[b0 + lane] : 0u;
    uint32_t inc = c;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t up = __shfl_up(inc, o);
      if (lane >= o) inc += up;
    }
    if (b0 + lane < nb) starts[b0 + lane] = acc + inc - c;
    acc += __shfl(inc, 63);
  }
  if (lane == 0) starts[nb] = acc;
}

// Cluster numbers of the starting rows, and every row without a label yet.
__global__ __launch_bounds__(kNumberBlock) void dbscan_number_kernel(
    int64_t n, const uint32_t* __restrict__ root, const uint32_t* __restrict__ starts,
    uint32_t* __restrict__ cid, uint32_t* __restrict__ label) {
  __shared__ uint32_t wave_at[kNumberBlock / 64];
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kNumberBlock + threadIdx.x;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const bool first = i < n && root[i] == static_cast<uint32_t>(i);
  const uint64_t m = __ballot(first);
  if (lane == 0) wave_at[w] = static_cast<uint32_t>(__popcll(m));
  __syncthreads();
  uint32_t at = starts[blockIdx.x];
  for (int v = 0; v < w; ++v) at += wave_at[v];
  if (first) cid[i] = at + static_cast<uint32_t>(__popcll(m & ((uint64_t(1) << lane) - 1)));
  if (i < n) label[i] = 0xffffffffu;
}

// A non-core row takes the lowest cluster among its core neighbours.
__global__ __launch_bounds__(256) void dbscan_border_kernel(const uint2* __restrict__ pairs,
                                                            unsigned long long cap,
                                                            const unsigned long long* __restrict__ cursor,
                                                            const uint32_t* __restrict__ root,
                                                            const uint32_t* __restrict__ cid,
                                                            uint32_t* __restrict__ label) {
  const unsigned long long m = min(*cursor, cap);
  for (unsigned long long e = static_cast<unsigned long long>(blockIdx.x) * blockDim.x + threadIdx.x;
       e < m; e += static_cast<unsigned long long>(gridDim.x) * blockDim.x) {
    const uint2 p = pairs[e];
    if (p.x == kNoRow) continue;
    const uint32_t rx = root[p.x], ry = root[p.y];
    if ((rx == 0xffffffffu) == (ry == 0xffffffffu)) continue;
    if (rx == 0xffffffffu)
      atomicMin(&label[p.x], cid[ry]);
    else
      atomicMin(&label[p.y], cid[rx]);
  }
}

__global__ void dbscan_labels_kernel(int64_t n, const uint32_t* __restrict__ root,
                                     const uint32_t* __restrict__ cid, uint32_t* __restrict__ label) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x)
    if (root[i] != 0xffffffffu) label[i] = cid[root[i]];  // others: a cluster, or -1
}

// The rows in the order of their groups, for one fit.
template <typename T>
struct GroupedRows {
  DevBuf rows, y2m, place, box;
  int64_t nt = 0;  // tiles, the padding between groups included

  void release() {
    rows.release();
    y2m.release();
    place.release();
    box.release();
  }
  // *ok is false, with no error, when the copy does not fit the memory: the
  // fit then takes every tile pair of the rows as they lie.
  int build(const T* src, int64_t n, int ld, int d, const double* src_y2m, hipStream_t s, bool* ok) {
    const int P = pivot_count(n), dims = std::min(d, kPivotDims);
    nt = n / kMR + P + 1;  // each group, the one of the rows left out too, ends in a partial tile
    const int64_t m = nt * kMR;
    DevBuf pivots, group, counts;
    if (m >= static_cast<int64_t>(kNoRow) || rows.alloc(sizeof(T) * m * ld, s) != hipSuccess ||
        y2m.alloc(sizeof(double) * m, s) != hipSuccess || place.alloc(sizeof(uint32_t) * m, s) != hipSuccess ||
        box.alloc(sizeof(double) * 2 * d * nt, s) != hipSuccess ||
        pivots.alloc(sizeof(double) * dims * P, s) != hipSuccess || group.alloc(n, s) != hipSuccess ||
        counts.alloc(sizeof(uint32_t) * 2 * (kMaxPivots + 1), s) != hipSuccess) {
      (void)hipGetLastError();
      release();
      *ok = false;
      return SC_OK;
    }
    uint32_t* sizes = counts.as<uint32_t>();
    uint32_t* pl = place.as<uint32_t>();
    SC_HIP(hipMemsetAsync(sizes, 0, sizeof(uint32_t) * 2 * (kMaxPivots + 1), s));
    ProfScope ps("dbscan_group", s);
    auto grid = [](int64_t threads, int block) {
      return dim3(static_cast<unsigned>(std::min<int64_t>((threads + block - 1) / block, 1 << 20)));
    };
    hipLaunchKernelGGL(dbscan_pivots_kernel<T>, grid(P * dims, 256), dim3(256), 0, s, src, n, ld, dims, P,
                       pivots.as<double>());
    hipLaunchKernelGGL(dbscan_empty_kernel, dim3(512), dim3(256), 0, s, m, pl);
    hipLaunchKernelGGL(dbscan_group_kernel<T>, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, s,
                       src, n, ld, dims, P, pivots.as<double>(), src_y2m, group.as<uint8_t>(), sizes);
    hipLaunchKernelGGL(dbscan_place_kernel,
                       dim3(static_cast<unsigned>((n + kPlaceThreads - 1) / kPlaceThreads)),
                       dim3(kPlaceThreads), 0, s, n, P, group.as<uint8_t>(), sizes, sizes + kMaxPivots + 1, pl);
    hipLaunchKernelGGL(dbscan_gather_kernel<T>, dim3(4096), dim3(256), 0, s, src, src_y2m, m, ld, pl,
                       rows.template as<T>(), y2m.template as<double>());
    hipLaunchKernelGGL(dbscan_boxes_kernel<T>, dim3(static_cast<unsigned>((nt * ld + 255) / 256)), dim3(256), 0,
                       s, rows.template as<T>(), y2m.template as<double>(), nt, ld, d, box.template as<double>());
    SC_HIP(hipGetLastError());
    *ok = true;
    return SC_OK;
  }
};

// The pair store of a fit: room for 64 neighbours a row (32 Mi pairs at
// least), or what an earlier try counted.
template <typename T>
int fit_pairs(const sc_index* index, double radius, double bound, size_t min_samples,
              int32_t* labels, size_t* num_classes, hipStream_t s) {
  const int64_t n = static_cast<int64_t>(index->n);
  const int ld = static_cast<int>(index->ld), d = static_cast<int>(index->d);
  const T* rows = static_cast<const T*>(index->rows);
  const Bound64 bd = bound64<T>(ld);
  DevBuf local;
  const double* y2m = nullptr;
  if (int rc = ensure_norms64(const_cast<sc_index*>(index), local, &y2m, s)) return rc;
  const int64_t nqt = (n + kMQ - 1) / kMQ;
  const int64_t total = nqt * (nqt + 1) / 2;
  const int64_t per = (total + 511) / 512;
  const int64_t nb = (n + kNumberBlock - 1) / kNumberBlock;
  const double all = 0.5 * static_cast<double>(n) * static_cast<double>(n);
  unsigned long long cap = static_cast<unsigned long long>(
      std::min(all, static_cast<double>(std::max<int64_t>(32 * n, int64_t(1) << 25))) + 1.0);
  DevBuf deg, par, root, cid, lab, starts, cur;
  SC_HIP(deg.alloc(sizeof(uint32_t) * n, s));
  SC_HIP(par.alloc(sizeof(uint32_t) * n, s));
  SC_HIP(root.alloc(sizeof(uint32_t) * n, s));
  SC_HIP(cid.alloc(sizeof(uint32_t) * n, s));
  SC_HIP(lab.alloc(sizeof(uint32_t) * n, s));
  SC_HIP(starts.alloc(sizeof(uint32_t) * (nb + 1), s));
  SC_HIP(cur.alloc(3 * sizeof(unsigned long long), s));  // pairs; items taken; tile pairs swept
  const unsigned g = static_cast<unsigned>(std::min<int64_t>(4096, (n + 255) / 256));
  GroupedRows<T> gr;
  bool grouped = false;
  if (n >= kGroupMinRows)
    if (int rc = gr.build(rows, n, ld, d, y2m, s, &grouped)) return rc;
  for (;;) {
    DevBuf pairs;
    hipError_t e = pairs.alloc(sizeof(uint2) * cap, s);
    if (e != hipSuccess && grouped) {  // the pairs come before the groups
      (void)hipGetLastError();
      gr.release();
      grouped = false;
      scratch_trim(s);
      e = pairs.alloc(sizeof(uint2) * cap, s);
    }
    SC_HIP(e);
    const uint32_t* place = grouped ? gr.place.template as<uint32_t>() : nullptr;
    uint2* pp = pairs.as<uint2>();
    unsigned long long* cp = cur.as<unsigned long long>();
    SC_HIP(hipMemsetAsync(cp, 0, 3 * sizeof(unsigned long long), s));
    hipLaunchKernelGGL(dbscan_self_kernel, dim3(g), dim3(256), 0, s, y2m, n, deg.as<uint32_t>(),
                       par.as<uint32_t>());
    {
      ProfScope ps("dbscan_pairs", s);
      if (grouped) {
        const int64_t items = gr.nt * ((gr.nt + kRun - 1) / kRun);
        // the box test's own sums are within (d + 2) 2^-53 of the distance
        const double apart = (bound * bd.up + bd.tiny) * (1.0 + 1e-12 + d * 4.5e-16);
        hipLaunchKernelGGL(dbscan_near_pairs_kernel<T>, dim3(512), dim3(kMT), 0, s, gr.rows.template as<T>(),
                           gr.nt, ld, d, gr.y2m.template as<double>(), gr.box.template as<double>(), bd,
                           bound, apart, items, pp, cap, cp, cp + 1, cp + 2);
      } else {
        hipLaunchKernelGGL(dbscan_pairs_kernel<T>, dim3(static_cast<unsigned>((total + per - 1) / per)),
                           dim3(kMT), 0, s, rows, n, ld, d, y2m, bd, bound, total, per, pp, cap, cp);
      }
      SC_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(dbscan_verify_kernel<T>, dim3(2048), dim3(256), 0, s,
                       grouped ? gr.rows.template as<T>() : rows, ld, radius, place, pp, cap, cp,
                       deg.as<uint32_t>());
    hipLaunchKernelGGL(dbscan_join_kernel, dim3(512), dim3(256), 0, s, pp, cap, cp, deg.as<uint32_t>(),
                       static_cast<uint64_t>(min_samples), kJoinSample, par.as<uint32_t>());
    hipLaunchKernelGGL(dbscan_compress_kernel, dim3(g), dim3(256), 0, s, n, par.as<uint32_t>());
    hipLaunchKernelGGL(dbscan_join_kernel, dim3(2048), dim3(256), 0, s, pp, cap, cp, deg.as<uint32_t>(),
                       static_cast<uint64_t>(min_samples), 1, par.as<uint32_t>());
    hipLaunchKernelGGL(dbscan_roots_kernel, dim3(static_cast<unsigned>(nb)), dim3(kNumberBlock), 0, s, n,
                       deg.as<uint32_t>(), static_cast<uint64_t>(min_samples), par.as<uint32_t>(),
                       root.as<uint32_t>(), starts.as<uint32_t>());
    hipLaunchKernelGGL(dbscan_scan_kernel, dim3(1), dim3(64), 0, s, starts.as<uint32_t>(), nb);
    hipLaunchKernelGGL(dbscan_number_kernel, dim3(static_cast<unsigned>(nb)), dim3(kNumberBlock), 0, s, n,
                       root.as<uint32_t>(), starts.as<uint32_t>(), cid.as<uint32_t>(), lab.as<uint32_t>());
    hipLaunchKernelGGL(dbscan_border_kernel, dim3(2048), dim3(256), 0, s, pp, cap, cp,
                       root.as<uint32_t>(), cid.as<uint32_t>(), lab.as<uint32_t>());
    hipLaunchKernelGGL(dbscan_labels_kernel, dim3(g), dim3(256), 0, s, n, root.as<uint32_t>(),
                       cid.as<uint32_t>(), lab.as<uint32_t>());
    SC_HIP(hipGetLastError());
    unsigned long long done[3] = {0, 0, 0};
    uint32_t clusters = 0;
    SC_HIP(hipMemcpyAsync(done, cp, sizeof(done), hipMemcpyDeviceToHost, s));
    SC_HIP(hipMemcpyAsync(&clusters, starts.as<uint32_t>() + nb, sizeof(clusters), hipMemcpyDeviceToHost, s));
    SC_HIP(hipStreamSynchronize(s));
    if (done[0] > cap) {  // denser than the store: once more with room for all
      cap = done[0];
      continue;
    }
    *num_classes = clusters;
    last_stats().queries = static_cast<uint64_t>(n);
    last_stats().candidates = (grouped ? done[2] : static_cast<uint64_t>(total)) * (kMQ * kMR);
    return download_staged(labels, lab.p, sizeof(uint32_t) * n, s);
  }
}

int check_metric(sc_metric metric, uint16_t p) {
  if (metric != SC_EUCLIDIAN && metric != SC_MANHATTAN && metric != SC_MINKOWSKI)
    return fail(SC_ERR_UNSUPPORTED, "unknown metric");
  if (metric == SC_MINKOWSKI && p < 1) return fail(SC_ERR_PANIC, "p must be at least 1");
  return SC_OK;
}

}  // namespace

extern "C" {

int sc_dbscan_fit(const sc_index* index, double eps, size_t min_samples, sc_metric metric,
                  uint16_t p, int32_t* labels, size_t* num_classes) {
  clear_error();
  if (!index || !labels || !num_classes) return fail(SC_PARAMETERS_ERROR, "null argument");
  *num_classes = 0;
  last_stats() = sc_stats{};
  // dbscan.rs:278-284
  if (min_samples < 1) return fail(SC_FIT_FAILED, "Invalid minPts");
  if (eps <= 0.0) return fail(SC_FIT_FAILED, "Invalid radius: ");
  if (int rc = check_metric(metric, p)) return rc;
  const size_t n = index->n;
  if (n == 0) return SC_OK;
  SC_HIP(hipSetDevice(index->device));
  hipStream_t s = stream_for(index);
  if (metric == SC_EUCLIDIAN) {
    // the radius search's conservative bound on the sum
    const double bound = eps * eps * (1.0 + 1e-12) + 1e-300;
    // (false for NaN, and for radii that sums overflowing the rows' type pass)
    if (index->dtype == SC_F64 ? bound < sum_limit<double>() : bound < sum_limit<float>()) {
      const int rc = index->dtype == SC_F64
                         ? fit_pairs<double>(index, eps, bound, min_samples, labels, num_classes, s)
                         : fit_pairs<float>(index, eps, bound, min_samples, labels, num_classes, s);
      if (rc != SC_ERR_OUT_OF_MEMORY) return rc;
      clear_error();  // the neighbour lists may fit
    }
  }
  sc_radius_result nb;
  // the expansion reads the neighbour rows only, not their distances
  if (int rc = radius_search_device(index, index->rows, static_cast<int64_t>(n), metric, p, eps,
                                    &nb, s, false))
    return rc;
  const size_t total = nb.idx.size();
  std::vector<uint32_t> root(n);
  {
    DevBuf doff, didx, dcore, dpar, droot;
    SC_HIP(doff.alloc(sizeof(uint64_t) * (n + 1), s));
    SC_HIP(didx.alloc(sizeof(int64_t) * std::max<size_t>(total, 1), s));
    SC_HIP(dcore.alloc(n, s));
    SC_HIP(dpar.alloc(sizeof(uint32_t) * n, s));
    SC_HIP(droot.alloc(sizeof(uint32_t) * n, s));
    if (int rc = upload_staged(doff.p, nb.offsets.data(), sizeof(uint64_t) * (n + 1), s)) return rc;
    if (int rc = upload_staged(didx.p, nb.idx.data(), sizeof(int64_t) * total, s)) return rc;
    const int64_t nn = static_cast<int64_t>(n);
    const unsigned g = static_cast<unsigned>(std::min<int64_t>(4096, (nn + 255) / 256));
    hipLaunchKernelGGL(dbscan_init_kernel, dim3(g), dim3(256), 0, s, doff.as<uint64_t>(), nn,
                       static_cast<uint64_t>(min_samples), dcore.as<uint8_t>(), dpar.as<uint32_t>());
    const unsigned gu = static_cast<unsigned>(std::min<int64_t>(8192, (nn + 3) / 4));
    hipLaunchKernelGGL(dbscan_union_kernel, dim3(gu), dim3(256), 0, s, doff.as<uint64_t>(),
                       didx.as<int64_t>(), nn, dcore.as<uint8_t>(), dpar.as<uint32_t>());
    hipLaunchKernelGGL(dbscan_root_kernel, dim3(g), dim3(256), 0, s, nn, dcore.as<uint8_t>(),
                       dpar.as<uint32_t>(), droot.as<uint32_t>());
    SC_HIP(hipGetLastError());
    if (int rc = download_staged(root.data(), droot.p, sizeof(uint32_t) * n, s)) return rc;
  }
  auto count = [&](size_t i) { return static_cast<size_t>(nb.offsets[i + 1] - nb.offsets[i]); };
  // clusters numbered by their smallest core row, in index order
  // (dbscan.rs:286-346: the outer loop starts a cluster there)
  std::vector<int32_t> cid(n, -1);
  int32_t k = 0;
  for (size_t i = 0; i < n; ++i)
    if (count(i) >= min_samples && root[i] == i) cid[i] = k++;
  std::vector<int32_t> y(n, -1);
  for (size_t i = 0; i < n; ++i) {
    if (count(i) >= min_samples) {
      y[i] = cid[root[i]];
      continue;
    }
    // a non-core row: the lowest cluster among its core neighbours
    int32_t best = -1;
    for (uint64_t e = nb.offsets[i]; e < nb.offsets[i + 1]; ++e) {
      const size_t j = static_cast<size_t>(nb.idx[e]);
      if (count(j) >= min_samples) {
        const int32_t c = cid[root[j]];
        if (best < 0 || c < best) best = c;
      }
    }
    y[i] = best;
  }
  std::copy(y.begin(), y.end(), labels);
  *num_classes = static_cast<size_t>(k);
  return SC_OK;
}

int sc_dbscan_predict(const sc_index* index, const int32_t* labels, size_t num_classes,
                      double eps, sc_metric metric, uint16_t p, const void* queries, size_t q,
                      int32_t* out) {
  clear_error();
  if (!index || !labels || !out || (!queries && q > 0))
    return fail(SC_PARAMETERS_ERROR, "null argument");
  // find_radius's own check (linear_search.rs:90-95)
  if (!(eps > 0.0)) return fail(SC_FIND_FAILED, "radius should be > 0");
  if (int rc = check_metric(metric, p)) return rc;
  if (q == 0) return SC_OK;
  SC_HIP(hipSetDevice(index->device));
  hipStream_t s = stream_for(index);
  sc_radius_result nb;
  {
    DevBuf dq;
    SC_HIP(dq.alloc(q * index->ld * elem_size(index->dtype), s));
    if (int rc = upload_padded(queries, index->dtype, q, index->d, index->ld, dq.p, s)) return rc;
    if (int rc = radius_search_device(index, dq.p, static_cast<int64_t>(q), metric, p, eps, &nb, s,
                                      false))
      return rc;
  }
  // dbscan.rs:368-393
  std::vector<size_t> hist(num_classes + 1);
  for (size_t i = 0; i < q; ++i) {
    std::fill(hist.begin(), hist.end(), 0);
    for (uint64_t e = nb.offsets[i]; e < nb.offsets[i + 1]; ++e) {
      const int32_t yi = labels[nb.idx[e]];
      if (yi < 0)
        hist[num_classes] += 1;
      else if (static_cast<size_t>(yi) < num_classes)
        hist[static_cast<size_t>(yi)] += 1;
      else
        return fail(SC_PARAMETERS_ERROR, "label out of range");
    }
    size_t which = 0, m = hist[0];
    for (size_t c = 1; c <= num_classes; ++c)
      if (hist[c] > m) {
        m = hist[c];
        which = c;
      }
    out[i] = which != num_classes ? static_cast<int32_t>(which + 1) : 0;
  }
  return SC_OK;
}

}  // extern "C"
