// Euclidian kNN in FP64 on the matrix cores (LinearKNNSearch::find,
// linear_search.rs:52-84) for f64 and f32 rows.
//
//   dense    The first rows (kDenseRows) of the index: L, the lower bound on
//            D of mfma64.hpp, of every (query, row), written out.
//   select0  One wavefront per query walks its L values in row order with
//            the k smallest upper bounds U seen so far across its lanes: a
//            row whose L is below the running k-th is a candidate.
//   scan     The rest in levels whose row ranges grow geometrically.  Each
//            row is tested against T, the k-th smallest U of all earlier
//            levels' candidates (at or above the k-th smallest S of the rows
//            before the level, hence at or above the heap's threshold), and
//            the rows below it go to a list per (query, piece), in row
//            order.  A piece that collects many candidates (rows sorted by
//            class, say) lowers T by its own k-th U as it goes, so lists stay
//            short for any order of the rows that the heap itself would not
//            thrash on.
//   select   The k smallest U so far, with the new level's candidates.
//   finish   One workgroup per query: S of every candidate in the
//            reference's arithmetic and order, then HeapSelection replayed
//            over them in row order.  A row that enters the reference heap
//            has S below the running k-th S of the earlier rows, so the
//            candidates are a superset of the entrants and every other row
//            would be a no-op: the heap array, order included, and the
//            distance bits are the reference's.
// Queries whose lists overflow, or whose norm is out of the bound's range,
// are recomputed by the sequential exact kernel.
//
// All arithmetic is FP64 (f32 rows are widened exactly); the bound's band is
// 1e-13 of the norms for f64 rows and 2e-7 of the distance for f32 rows, so
// hardly a row is tested in vain.
//
// The scan uses 64 % of the FP64 matrix rate (72 TFLOP/s in a large matrix
// product on this card) at 64 dimensions and 76 % at 100; mfma64.hpp has what
// bounds it.  4,096 queries x 200,000 x 64 f64 rows take 2.42 ms (12.8 ms with
// a tile of vector subtract, multiply, add), 3,001 x 750,000 x 100 f32 8.1 ms
// (42.0), 55 TFLOP/s.  The prefix is 1,024 rows because its selection
// is a walk per query; two levels then leave about 250 candidates per query
// at k = 10, and one more level would cost two launches to save 100.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

#include "common.hpp"
#include "heap.hpp"
#include "metric.hpp"
#include "knn_lists.hpp"
#include "mfma64.hpp"

namespace sc {

// from knn_exact.hip
int launch_serial_exact(const sc_index* index, const void* d_queries, int k, const uint32_t* list,
                        const uint32_t* list_n, int64_t* d_idx, double* d_dist, uint32_t* d_count,
                        hipStream_t stream);

namespace {


// Sixteen lanes per row: the squared norm (any order: the gap covers it).
template <typename T>
__device__ __forceinline__ double row_norm(const T* __restrict__ r, int ld, int sub, bool* finite) {
  double s = 0.0;
  bool ok = true;
  for (int j = sub; j < ld; j += 16) {
    const double v = static_cast<double>(r[j]);
    ok = ok && isfinite(v);
    s += v * v;
  }
#pragma unroll
  for (int o = 8; o >= 1; o >>= 1) {
    s += __shfl_xor(s, o, 16);
    ok = (__shfl_xor(static_cast<int>(ok), o, 16) != 0) && ok;
  }
  *finite = ok;
  return s;
}

template <typename T>
__global__ void row_norms_kernel(const T* __restrict__ rows, int64_t n, int64_t npad, int ld,
                                 double shrink, double* __restrict__ y2m) {
  const int sub = threadIdx.x & 15;
  for (int64_t i = lane_row(16); i < npad; i += lane_row_step(16)) {  // sixteen lanes together
    double out = INFINITY;
    if (i < n) {
      bool finite;
      const double s = row_norm(rows + i * ld, ld, sub, &finite);
      if (finite) out = s < kNorm64Limit ? s * shrink : NAN;
    }
    if (sub == 0) y2m[i] = out;
  }
}

template <typename T>
__global__ void query_norms_kernel(const T* __restrict__ qs, int64_t q, int ld, double shrink,
                                   double* __restrict__ x2m, uint32_t* __restrict__ list,
                                   uint32_t* __restrict__ list_n) {
  const int sub = threadIdx.x & 15;
  for (int64_t i = lane_row(16); i < q; i += lane_row_step(16)) {
    bool finite;
    const double s = row_norm(qs + i * ld, ld, sub, &finite);
    if (sub != 0) continue;
    const bool in = finite && s < kNorm64Limit;
    x2m[i] = in ? s * shrink : INFINITY;
    if (finite && !in) list[atomicAdd(list_n, 1u)] = static_cast<uint32_t>(i);
  }
}

// L of queries x the first `cols` rows (a multiple of kMR, rows past the
// index +inf), row-major by query.  One workgroup per (query tile, row tile).
template <typename T>
__global__ __launch_bounds__(kMT, 2) void dense_kernel(const T* __restrict__ rows, int64_t n,
                                                       int ld, int d,
                                                       const double* __restrict__ y2m,
                                                       const T* __restrict__ queries, int64_t q,
                                                       const double* __restrict__ x2m,
                                                       int64_t cols, double* __restrict__ out) {
  __shared__ MSmem sm;
  __shared__ double sx[kMQ];
  const int64_t q0 = static_cast<int64_t>(blockIdx.x) * kMQ;
  const int64_t tile = blockIdx.y;
  const int tid = threadIdx.x;
  if (tid < kMQ) sx[tid] = x2m[min(q0 + tid, q - 1)];
  mfma64_sweep<T, true>(sm, rows, n, ld, d, y2m, queries, q, q0, 0, tile, tile + 1,
                        [&](int64_t t, MAcc& acc, int par) {
    const MLane ml;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int rl = 16 * i + ml.lr;
      const double y = sm.y2[par][rl];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int ql = ml.wave * 32 + 16 * j + 4 * v + ml.lg;
          if (q0 + ql < q) out[(q0 + ql) * cols + t * kMR + rl] = acc[i][j][v] + (sx[ql] + y);
        }
    }
  });
}

__global__ __launch_bounds__(64 * kSelectWaves) void select_dense_kernel(
    const double* __restrict__ L, int64_t cols, const double* __restrict__ y2m,
    const double* __restrict__ x2m, int64_t q, int k, Bound64 bd, int cap,
    uint32_t* __restrict__ cand_idx, uint32_t* __restrict__ cand_count, double* __restrict__ seed) {
  const int lane = threadIdx.x & 63;
  const int64_t qi = static_cast<int64_t>(blockIdx.x) * kSelectWaves + (threadIdx.x >> 6);
  if (qi >= q) return;  // the whole wave
  const double x2 = x2m[qi];
  KSmallest<double> ks;
  ks.clear();
  uint32_t cnt = 0;
  const double* l = L + qi * cols;
  if (x2 < INFINITY) {
    double lv = l[lane], yv = y2m[lane];
    // (past cap, the query's list is lost; what was seen stays a bound)
    for (int64_t c0 = 0; c0 < cols && cnt <= static_cast<uint32_t>(cap); c0 += 64) {
      const double cl = lv, cy = yv;
      if (c0 + 64 < cols) {  // the next chunk's loads run under this one's work
        lv = l[c0 + 64 + lane];
        yv = y2m[c0 + 64 + lane];
      }
      const double u = sum_upper(bd, cl, x2 + cy);
      const bool live = !(cy == INFINITY);
      // below the running k-th (on D's scale); NaN stays a candidate
      double th = ks.kth < INFINITY ? ks.kth * bd.up + bd.tiny : INFINITY;
      uint64_t m = __ballot(live && !(cl >= th));
      while (m) {
        const int src = __builtin_ctzll(m);
        if (cnt < static_cast<uint32_t>(cap) && lane == 0)
          cand_idx[qi * cap + cnt] = static_cast<uint32_t>(c0 + src);
        ++cnt;
        const double x = lane_value(u, src);
        m &= m - 1;
        if (x < ks.kth) {
          ks.insert(x, lane, k);
          th = ks.kth < INFINITY ? ks.kth * bd.up + bd.tiny : INFINITY;
          m &= __ballot(live && !(cl >= th));
        }
      }
    }
  }
  if (lane < k) seed[qi * k + lane] = ks.b;
  if (lane == 0) cand_count[qi] = cnt;
}

template <typename T>
__global__ __launch_bounds__(kMT, 2) void scan_kernel(
    const T* __restrict__ rows, int64_t n, int ld, int d, const double* __restrict__ y2m,
    const T* __restrict__ queries, int64_t q, const double* __restrict__ x2m,
    const double* __restrict__ seed, int k, Bound64 bd, Level lv, ScanOut<double> out) {
  __shared__ MSmem sm;
  const MLane ml;
  const int64_t nqt = (q + kMQ - 1) / kMQ;
  const uint32_t grow = static_cast<uint32_t>(max(2 * k, 32));
  int64_t pos = static_cast<int64_t>(blockIdx.x) * lv.per;
  const int64_t end = min(pos + lv.per, nqt * lv.tiles);
  while (pos < end) {
    const int64_t qt = pos / lv.tiles;
    const int64_t tb = pos - qt * lv.tiles;
    const int64_t te = min(lv.tiles, tb + (end - pos));
    const int list = static_cast<int>(blockIdx.x - qt * lv.tiles / lv.per);
    const int64_t q0 = qt * kMQ;
    // the lane's two queries: norm, threshold, entries so far and at the
    // last look (the same in all four lanes of a column)
    double x2[2], th[2];
    uint32_t cnt[2] = {0u, 0u}, mark[2] = {0u, 0u};
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t qi = q0 + ml.query_of(j);
      x2[j] = qi < q ? x2m[qi] : INFINITY;
      // queries that take no part: nothing is below -inf
      th[j] = x2[j] < INFINITY ? acc_threshold(bd, seed[qi * k + k - 1], x2[j]) : -INFINITY;
    }
    auto slot_of = [&](int ql, uint32_t c) {
      return (q0 + ql) * out.entries + lv.entry0 + static_cast<int64_t>(list) * lv.cap + c;
    };
    mfma64_sweep<T, false>(sm, rows, n, ld, d, y2m, queries, q, q0, lv.row0, tb, te,
                           [&](int64_t t, MAcc& acc, int par) {
      const int64_t r0 = lv.row0 + t * kMR;
      tile_hits(ml, acc, th, sm.y2[par], [&](int i, int j, int v, int rl, bool hit, uint64_t m) {
        m &= ml.column();
        const uint32_t c = cnt[j] + __popcll(m & ml.below());
        if (hit && c < static_cast<uint32_t>(lv.cap)) {
          const int64_t s = slot_of(ml.query_of(j), c);
          out.idx[s] = static_cast<uint32_t>(r0 + rl);
          out.u[s] = sum_upper(bd, acc[i][j][v] + x2[j], x2[j] + sm.y2[par][rl]);
        }
        cnt[j] += __popcll(m);
      });
      // lists that grew by `grow` since they were last looked at: their own
      // k-th U is a threshold too
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        uint64_t g = __ballot(cnt[j] - mark[j] >= grow) & 0xffffu;
        while (g) {
          const int src = __builtin_ctzll(g);  // the column
          g &= g - 1;
          const uint32_t c = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(cnt[j]), src));
          if (c > static_cast<uint32_t>(lv.cap)) {
            // its list is lost (the sequential kernel takes the query): no
            // more rows for it
            if (ml.lr == src) {
              th[j] = -INFINITY;
              mark[j] = c;
            }
            continue;
          }
          const uint32_t m = c;
          const double* u = out.u + slot_of(ml.wave * 32 + 16 * j + src, 0);
          // entries that other lanes of this wavefront stored
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
          KSmallest<double> ks;
          ks.clear();
          ks.take(u, m, ml.lane, k);
          if (ml.lr == src) {
            const double lower = acc_threshold(bd, ks.kth, x2[j]);
            if (lower < th[j]) th[j] = lower;
            mark[j] = c;
          }
        }
      }
    });
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t qi = q0 + ml.query_of(j);
      if (ml.lg == 0 && qi < q) out.count[qi * out.lists + lv.list0 + list] = cnt[j];
    }
    pos += te - tb;
    __syncthreads();  // the sweep's LDS is staged anew
  }
}

template <typename T>
int run_f64(const sc_index* index, const T* d_queries, int64_t q, int k, int64_t* d_idx,
            double* d_dist, uint32_t* d_count, hipStream_t s, sc_stats* stats) {
  const int64_t n = static_cast<int64_t>(index->n);
  const int ld = static_cast<int>(index->ld), d = static_cast<int>(index->d);
  const T* rows = static_cast<const T*>(index->rows);
  const Bound64 bd = bound64<T>(ld);
  DevBuf local;
  const double* y2m = nullptr;
  if (int rc = ensure_norms64(const_cast<sc_index*>(index), local, &y2m, s)) return rc;

  const int64_t cols = std::min<int64_t>(kDenseRows, (n + kMR - 1) / kMR * kMR);
  const std::vector<int64_t> edge = level_edges(n, cols);
  const int nlev = static_cast<int>(edge.size()) - 1;
  const int pre_cap = static_cast<int>(std::min<int64_t>(
      cols, static_cast<int64_t>(3.0 * expected_entrants(k, static_cast<double>(cols))) + 64));
  // two workgroups per CU fit (LDS and registers)
  auto plan = [&](int64_t qn, Level (&lv)[kMaxLevels], ScanOut<double>& o) {
    plan_levels(edge, qn, kMQ, 512, k, lv, o);
  };
  Lists<double> ls{};
  ls.nlevels = nlev;
  ls.pre_cap = pre_cap;
  const Batches batches = plan_batches<double>(
      q, plan,
      [&](const ScanOut<double>& o) {
        return 12.0 * o.entries + 4.0 * o.lists + 4.0 * pre_cap + 8.0 * (cols + k + 1);
      },
      ls.lv, ls.out);
  const int64_t qb = batches.queries;
  DevBuf flags, olist, x2m, dense, pidx, pcnt, cidx, cu, ccnt, seed;
  SC_HIP(flags.alloc(64, s));  // [0] listed queries, [2..3] candidate total (u64)
  SC_HIP(olist.alloc(sizeof(uint32_t) * qb, s));
  SC_HIP(x2m.alloc(sizeof(double) * qb, s));
  SC_HIP(dense.alloc(sizeof(double) * qb * cols, s));
  SC_HIP(pidx.alloc(sizeof(uint32_t) * qb * pre_cap, s));
  SC_HIP(pcnt.alloc(sizeof(uint32_t) * qb, s));
  SC_HIP(seed.alloc(sizeof(double) * qb * k, s));
  SC_HIP(cidx.alloc(sizeof(uint32_t) * batches.entries, s));
  SC_HIP(cu.alloc(sizeof(double) * batches.entries, s));
  SC_HIP(ccnt.alloc(sizeof(uint32_t) * batches.lists, s));
  uint32_t* list_n = flags.as<uint32_t>();
  unsigned long long* total = reinterpret_cast<unsigned long long*>(flags.as<char>() + 8);
  hipLaunchKernelGGL(zero_words_kernel, dim3(1), dim3(64), 0, s, flags.as<uint32_t>(), int64_t{16});
  for (int64_t b0 = 0; b0 < q; b0 += qb) {
    const int64_t qn = std::min(qb, q - b0);
    const T* qs = d_queries + b0 * ld;
    if (qn != qb) plan(qn, ls.lv, ls.out);
    ls.pre_idx = pidx.as<uint32_t>();
    ls.pre_count = pcnt.as<uint32_t>();
    ls.out.idx = cidx.as<uint32_t>();
    ls.out.u = cu.as<double>();
    ls.out.count = ccnt.as<uint32_t>();
    hipLaunchKernelGGL(zero_words_kernel, dim3(1), dim3(64), 0, s, list_n, int64_t{1});
    if (int rc = query_norms64<T>(qs, qn, ld, x2m.as<double>(), olist.as<uint32_t>(), list_n, s)) return rc;
    const unsigned nqt = static_cast<unsigned>((qn + kMQ - 1) / kMQ);
    const unsigned sel = static_cast<unsigned>((qn + kSelectWaves - 1) / kSelectWaves);
    {
      ProfScope ps("knn_scan", s);
      hipLaunchKernelGGL(dense_kernel<T>, dim3(nqt, static_cast<unsigned>(cols / kMR)), dim3(kMT), 0,
                         s, rows, n, ld, d, y2m, qs, qn, x2m.as<double>(), cols, dense.as<double>());
      hipLaunchKernelGGL(select_dense_kernel, dim3(sel), dim3(64 * kSelectWaves), 0, s,
                         dense.as<double>(), cols, y2m, x2m.as<double>(), qn, k, bd, pre_cap,
                         pidx.as<uint32_t>(), pcnt.as<uint32_t>(), seed.as<double>());
      SC_HIP(hipGetLastError());
      if (nlev > 0) {
        // pieces that a level does not have leave empty lists
        const int64_t w = qn * ls.out.lists;
        hipLaunchKernelGGL(zero_words_kernel, dim3(static_cast<unsigned>(std::min<int64_t>(1024, (w + 255) / 256))),
                           dim3(256), 0, s, ls.out.count, w);
      }
      for (int i = 0; i < nlev; ++i) {
        hipLaunchKernelGGL(scan_kernel<T>, dim3(static_cast<unsigned>(ls.lv[i].groups)), dim3(kMT), 0,
                           s, rows, n, ld, d, y2m, qs, qn, x2m.as<double>(), seed.as<double>(), k, bd,
                           ls.lv[i], ls.out);
        if (i + 1 < nlev)
          hipLaunchKernelGGL(select_level_kernel<double>, dim3(sel), dim3(64 * kSelectWaves), 0, s, ls.lv[i],
                             ls.out, qn, k, seed.as<double>());
        SC_HIP(hipGetLastError());
      }
    }
    {
      ProfScope ps("knn_replay", s);
      launch_finish<T, kEuclid>(rows, ld, qs, qn, k, ls, d_idx + b0 * k, d_dist + b0 * k, d_count + b0,
                                olist.as<uint32_t>(), list_n, stats ? total : nullptr, s);
      SC_HIP(hipGetLastError());
    }
    if (int rc = launch_serial_exact(index, qs, k, olist.as<uint32_t>(), list_n, d_idx + b0 * k,
                                     d_dist + b0 * k, d_count + b0, s))
      return rc;
    if (stats && !(qn == q && defer_search_counters(flags.p, s))) {
      uint64_t h[2] = {0, 0};
      SC_HIP(hipMemcpyAsync(h, flags.p, 16, hipMemcpyDeviceToHost, s));
      SC_HIP(hipStreamSynchronize(s));
      stats->overflow_queries += static_cast<uint32_t>(h[0]);
      if (b0 + qn >= q) stats->candidates += h[1];
    }
  }
  if (stats) stats->queries += static_cast<uint64_t>(q);
  return SC_OK;
}

}  // namespace

int ensure_norms64(sc_index* ix, DevBuf& local, const double** y2m, hipStream_t s) {
  const int64_t n = static_cast<int64_t>(ix->n);
  const int64_t npad = std::max<int64_t>(kMR, (n + kMR - 1) / kMR * kMR);
  const int ld = static_cast<int>(ix->ld);
  const double shrink = 1.0 - norm_gap(ld);
  auto launch = [&](double* out) -> int {
    const dim3 grid(row_blocks(npad, 16, 256));
    if (ix->dtype == SC_F64)
      hipLaunchKernelGGL(row_norms_kernel<double>, grid, dim3(256), 0, s,
                         static_cast<const double*>(ix->rows), n, npad, ld, shrink, out);
    else
      hipLaunchKernelGGL(row_norms_kernel<float>, grid, dim3(256), 0, s,
                         static_cast<const float*>(ix->rows), n, npad, ld, shrink, out);
    SC_HIP(hipGetLastError());
    return SC_OK;
  };
  const bool capturing = stream_capturing(s);
  std::lock_guard<std::mutex> lk(*static_cast<std::mutex*>(ix->mu));
  if (ix->norms64 && !ix->norms64_ready) {
    // (a query is not an operation of the stream: it is allowed beside a capture)
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    const bool swapped = capturing && hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
    if (!capturing || swapped) {
      ix->norms64_ready = hipEventQuery(ix->norms64_done) == hipSuccess;
      if (!ix->norms64_ready) (void)hipGetLastError();  // not ready is no error
    }
    if (swapped) (void)hipThreadExchangeStreamCaptureMode(&mode);
  }
  if (ix->norms64 && (ix->norms64_ready || (!capturing && s == ix->norms64_stream))) {
    // (a new stream may have got the handle of the one that built them)
    if (!ix->norms64_ready) SC_HIP(hipStreamWaitEvent(s, ix->norms64_done, 0));
    *y2m = ix->norms64;
    return SC_OK;
  }
  if (ix->norms64 || capturing) {
    SC_HIP(local.alloc(sizeof(double) * npad, s));
    if (int rc = launch(local.as<double>())) return rc;
    *y2m = local.as<double>();
    return SC_OK;
  }
  double* p = nullptr;
  SC_HIP(hipMalloc(reinterpret_cast<void**>(&p), sizeof(double) * npad));
  hipEvent_t done = nullptr;
  hipError_t e = hipEventCreateWithFlags(&done, hipEventDisableTiming);
  int rc = e == hipSuccess ? launch(p) : hip_fail(e, "row norms");
  if (rc == SC_OK && (e = hipEventRecord(done, s)) != hipSuccess) {
    rc = hip_fail(e, "row norms");
    (void)hipStreamSynchronize(s);  // p is freed below
  }
  if (rc != SC_OK) {
    if (done) (void)hipEventDestroy(done);
    (void)hipFree(p);
    return rc;
  }
  ix->norms64 = p;
  ix->norms64_done = done;
  ix->norms64_stream = s;
  *y2m = p;
  return SC_OK;
}

template <typename T>
int query_norms64(const T* queries, int64_t q, int ld, double* x2m, uint32_t* list,
                  uint32_t* list_n, hipStream_t s) {
  hipLaunchKernelGGL(query_norms_kernel<T>, dim3(row_blocks(q, 16, 256)), dim3(256),
                     0, s, queries, q, ld, 1.0 - norm_gap(ld), x2m, list, list_n);
  SC_HIP(hipGetLastError());
  return SC_OK;
}
template int query_norms64<double>(const double*, int64_t, int, double*, uint32_t*, uint32_t*, hipStream_t);
template int query_norms64<float>(const float*, int64_t, int, double*, uint32_t*, uint32_t*, hipStream_t);

int knn_f64_device(const sc_index* index, const void* d_queries, int64_t q, int k, int64_t* d_idx,
                   double* d_dist, uint32_t* d_count, hipStream_t stream, sc_stats* stats) {
  if (index->dtype == SC_F64)
    return run_f64(index, static_cast<const double*>(d_queries), q, k, d_idx, d_dist, d_count,
                   stream, stats);
  return run_f64(index, static_cast<const float*>(d_queries), q, k, d_idx, d_dist, d_count, stream,
                 stats);
}

}  // namespace sc
