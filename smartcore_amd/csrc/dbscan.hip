// DBSCAN::fit and DBSCAN::predict (cluster/dbscan.rs:274-397) over a device
// index.
//
// The distance work -- find_radius (linear_search.rs:89-108) of every row,
// O(n^2 d) -- runs as one batched device radius search (each row's
// neighbours in index order, which is exactly the list find_radius returns).
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
// is its smallest row); the numbering and the non-core rows (whose lists are
// shorter than min_samples) are done on the host.  predict searches its
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

// The root of v's tree, halving the path on the way.  parent[x] <= x holds
// for every value ever stored, so reads that are stale still point at an
// ancestor, and the walk strictly decreases until it meets a root.
__device__ uint32_t dbscan_rep(uint32_t* parent, uint32_t v) {
  uint32_t cur = parent[v];
  if (cur != v) {
    uint32_t prev = v, next;
    while (cur > (next = parent[cur])) {
      parent[prev] = next;
      prev = cur;
      cur = next;
    }
  }
  return cur;
}

// Joins the trees of u and v: the larger root is linked to the smaller by a
// compare-and-swap; a failed swap returns a smaller value to continue from,
// so the loop ends.
__device__ void dbscan_link(uint32_t* parent, uint32_t u, uint32_t v) {
  uint32_t ru = dbscan_rep(parent, u), rv = dbscan_rep(parent, v);
  while (ru != rv) {
    if (ru < rv) {
      const uint32_t old = atomicCAS(&parent[rv], rv, ru);
      if (old == rv) break;
      rv = old;
    } else {
      const uint32_t old = atomicCAS(&parent[ru], ru, rv);
      if (old == ru) break;
      ru = old;
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
// reference's sum and counts both ends' neighbours; `union` joins the core
// rows of the remaining pairs; clusters are numbered by their smallest core
// row with a prefix sum, and a pair with one core end offers its cluster to
// the other.  Nothing but the labels goes to the host.  At 200,000 x 8 rows
// with 55 neighbours each, a fit took 91 ms (the search 73 ms, the lists and
// their trips over PCIe the rest) and takes 12.7 (the sweep 10.9, the union
// 2.0).

constexpr int kPairBuf = 128;  // pairs staged in LDS per wavefront

__device__ __forceinline__ int64_t triangle_row(int64_t pos) {
  int64_t r = static_cast<int64_t>((sqrt(8.0 * static_cast<double>(pos) + 1.0) - 1.0) * 0.5);
  while (r * (r + 1) / 2 > pos) --r;
  while ((r + 1) * (r + 2) / 2 <= pos) ++r;
  return r;
}

// Tiles (qt, t <= qt) numbered qt (qt + 1) / 2 + t, dealt to the workgroups
// in contiguous runs.  Each wavefront collects its pairs in an LDS buffer
// (a place is the buffer's fill plus the lane's rank in the hit mask) and
// empties it when the next mask may not fit, with one update of the global
// counter; pairs past cap are counted only.
template <typename T>
__global__ __launch_bounds__(kMT, 2) void dbscan_pairs_kernel(
    const T* __restrict__ rows, int64_t n, int ld, int d, const double* __restrict__ y2m, Bound64 bd,
    double bound, int64_t total, int64_t per, uint2* __restrict__ pairs, unsigned long long cap,
    unsigned long long* __restrict__ cursor) {
  __shared__ MSmem sm;
  __shared__ uint2 buf[kMT / 64][kPairBuf];
  const MLane ml;
  uint2* mine = buf[ml.wave];
  uint32_t fill = 0;  // the same in the whole wavefront
  auto flush = [&]() {
    unsigned long long base = 0;
    if (ml.lane == 0) base = atomicAdd(cursor, static_cast<unsigned long long>(fill));
    base = __shfl(base, 0);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    for (uint32_t e = ml.lane; e < fill; e += 64)
      if (base + e < cap) pairs[base + e] = mine[e];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    fill = 0;
  };
  int64_t pos = static_cast<int64_t>(blockIdx.x) * per;
  const int64_t end = min(pos + per, total);
  while (pos < end) {
    const int64_t qt = triangle_row(pos);
    const int64_t tb = pos - qt * (qt + 1) / 2;
    const int64_t te = min(qt + 1, tb + (end - pos));
    const int64_t q0 = qt * kMQ;
    double th[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const double x2 = y2m[q0 + ml.query_of(j)];
      // rows left out take no part; rows past the bound's range (NaN) pass
      // every test
      th[j] = x2 == INFINITY ? -INFINITY : acc_threshold(bd, bound, x2);
    }
    mfma64_sweep<T, false>(sm, rows, n, ld, d, y2m, rows, n, q0, 0, tb, te,
                           [&](int64_t t, MAcc& acc, int par) {
      tile_hits(ml, acc, th, sm.y2[par], [&](int, int j, int, int rl, bool hit, uint64_t m) {
        if (t == qt) {  // the diagonal tile: smaller rows only
          hit = hit && rl < ml.query_of(j);
          m = __ballot(hit);
        }
        const uint32_t c = static_cast<uint32_t>(__popcll(m));
        if (fill + c > kPairBuf) flush();
        if (hit)
          mine[fill + __popcll(m & ml.below())] =
              make_uint2(static_cast<uint32_t>(q0 + ml.query_of(j)), static_cast<uint32_t>(t * kMR + rl));
        fill += c;
      });
    });
    pos += te - tb;
    __syncthreads();  // the sweep's LDS is staged anew
  }
  flush();
}

// Decides each pair with the reference's distance: its ends' neighbour
// counts, or (no neighbours) an empty pair.
template <typename T>
__global__ __launch_bounds__(256) void dbscan_verify_kernel(const T* __restrict__ rows, int ld,
                                                            double radius, uint2* __restrict__ pairs,
                                                            unsigned long long cap,
                                                            const unsigned long long* __restrict__ cursor,
                                                            uint32_t* __restrict__ degree) {
  const unsigned long long m = min(*cursor, cap);
  for (unsigned long long e = static_cast<unsigned long long>(blockIdx.x) * blockDim.x + threadIdx.x;
       e < m; e += static_cast<unsigned long long>(gridDim.x) * blockDim.x) {
    const uint2 p = pairs[e];
    const double s = exact_sum<T, kEuclid>(rows + static_cast<int64_t>(p.x) * ld, rows + static_cast<int64_t>(p.y) * ld, ld);
    if (__builtin_sqrt(s) <= radius) {
      atomicAdd(&degree[p.x], 1u);
      atomicAdd(&degree[p.y], 1u);
    } else {
      pairs[e].x = 0xffffffffu;
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

__global__ __launch_bounds__(256) void dbscan_join_kernel(const uint2* __restrict__ pairs,
                                                          unsigned long long cap,
                                                          const unsigned long long* __restrict__ cursor,
                                                          const uint32_t* __restrict__ degree,
                                                          uint64_t min_samples, uint32_t* parent) {
  const unsigned long long m = min(*cursor, cap);
  for (unsigned long long e = static_cast<unsigned long long>(blockIdx.x) * blockDim.x + threadIdx.x;
       e < m; e += static_cast<unsigned long long>(gridDim.x) * blockDim.x) {
    const uint2 p = pairs[e];
    if (p.x != 0xffffffffu && degree[p.x] >= min_samples && degree[p.y] >= min_samples)
      dbscan_link(parent, p.x, p.y);
  }
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
    if (p.x == 0xffffffffu) continue;
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
  SC_HIP(cur.alloc(sizeof(unsigned long long), s));
  const unsigned g = static_cast<unsigned>(std::min<int64_t>(4096, (n + 255) / 256));
  for (;;) {
    DevBuf pairs;
    SC_HIP(pairs.alloc(sizeof(uint2) * cap, s));
    uint2* pp = pairs.as<uint2>();
    unsigned long long* cp = cur.as<unsigned long long>();
    SC_HIP(hipMemsetAsync(cp, 0, sizeof(unsigned long long), s));
    hipLaunchKernelGGL(dbscan_self_kernel, dim3(g), dim3(256), 0, s, y2m, n, deg.as<uint32_t>(),
                       par.as<uint32_t>());
    {
      ProfScope ps("dbscan_pairs", s);
      hipLaunchKernelGGL(dbscan_pairs_kernel<T>, dim3(static_cast<unsigned>((total + per - 1) / per)),
                         dim3(kMT), 0, s, rows, n, ld, d, y2m, bd, bound, total, per, pp, cap, cp);
      SC_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(dbscan_verify_kernel<T>, dim3(2048), dim3(256), 0, s, rows, ld, radius, pp, cap,
                       cp, deg.as<uint32_t>());
    hipLaunchKernelGGL(dbscan_join_kernel, dim3(2048), dim3(256), 0, s, pp, cap, cp, deg.as<uint32_t>(),
                       static_cast<uint64_t>(min_samples), par.as<uint32_t>());
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
    unsigned long long found = 0;
    uint32_t clusters = 0;
    SC_HIP(hipMemcpyAsync(&found, cp, sizeof(found), hipMemcpyDeviceToHost, s));
    SC_HIP(hipMemcpyAsync(&clusters, starts.as<uint32_t>() + nb, sizeof(clusters), hipMemcpyDeviceToHost, s));
    SC_HIP(hipStreamSynchronize(s));
    if (found > cap) {  // denser than the store: once more with room for all
      cap = found;
      continue;
    }
    *num_classes = clusters;
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
    if (index->dtype == SC_F64 ? bound < sum_limit<double>() : bound < sum_limit<float>())
      return index->dtype == SC_F64
                 ? fit_pairs<double>(index, eps, bound, min_samples, labels, num_classes, s)
                 : fit_pairs<float>(index, eps, bound, min_samples, labels, num_classes, s);
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
