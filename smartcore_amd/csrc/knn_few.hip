// LinearKNNSearch::find (linear_search.rs:52-84) for few queries over few
// rows: two launches.
//
// Such a call is bound by its launches and the chain between them, not by
// arithmetic: the matrix form (knn_f64.hip) takes nine, and its bounds,
// thresholds and lists save distances that cost next to nothing here.  So
//   sums     every pair's distance in the reference's arithmetic, a lane per
//            row, written out (64 rows per wavefront, through LDS);
//   replay   one wavefront per query reads them in row order, 1,024 at a time
//            with the next 1,024 on their way, and pushes those below the
//            heap's top, which is LinearKNNSearch's own loop.
// 1 query x 10,000 x 32 f64, k = 5, from host arrays: 83 us with the
// matrix form, 48 with this.
#include <hip/hip_runtime.h>

#include "common.hpp"
#include "heap.hpp"
#include "metric.hpp"

namespace sc {
namespace {

constexpr int kFewThreads = 256;
constexpr int kFewLoads = 16;
constexpr int64_t kFewChunk = 64 * kFewLoads;  // distances the replay takes at a time

// Rows n .. npad - 1 get +inf, which enters no heap.
template <typename T, int M>
__global__ __launch_bounds__(kFewThreads) void few_sums_kernel(const T* __restrict__ rows, int64_t n,
                                                               int64_t npad, int ld,
                                                               const T* __restrict__ queries,
                                                               double* __restrict__ dist) {
  extern __shared__ __align__(16) unsigned char few_smem[];
  T* qrow = reinterpret_cast<T*>(few_smem);
  __shared__ __align__(16) unsigned char tiles[kFewThreads / 64][kSumTileBytes];
  const int64_t qi = blockIdx.y;
  const int tid = threadIdx.x;
  for (int j = tid; j < ld; j += kFewThreads) qrow[j] = queries[qi * ld + j];
  __syncthreads();
  const int64_t r = static_cast<int64_t>(blockIdx.x) * kFewThreads + tid;
  const double s = wave_exact_sums<T, M>(qrow, rows, static_cast<uint32_t>(min(r, n - 1)), ld, tiles[tid >> 6]);
  const double dv = finalize<M>(s, 1.0);
  if (r < npad) dist[qi * npad + r] = r < n ? dv : INFINITY;
}

__global__ __launch_bounds__(64) void few_replay_kernel(const double* __restrict__ dist, int64_t npad, int k,
                                                        int64_t* __restrict__ out_idx,
                                                        double* __restrict__ out_dist,
                                                        uint32_t* __restrict__ out_count) {
  const int lane = threadIdx.x;
  const int64_t qi = blockIdx.x;
  const double* d = dist + qi * npad + lane;
  double v[kFewLoads], w[kFewLoads];
#pragma unroll
  for (int u = 0; u < kFewLoads; ++u) v[u] = d[64 * u];
  double hd = INFINITY, top = INFINITY;
  asm volatile("" : "+v"(hd), "+v"(top));  // (a uniform 64-bit literal would lose its upper half)
  uint32_t hi = 0xffffffffu;
  for (int64_t r0 = 0; r0 < npad; r0 += kFewChunk) {
    if (r0 + kFewChunk < npad) {
#pragma unroll
      for (int u = 0; u < kFewLoads; ++u) w[u] = d[r0 + kFewChunk + 64 * u];
    }
#pragma unroll
    for (int u = 0; u < kFewLoads; ++u) {
      uint64_t b = __ballot(v[u] < top);
      while (b) {
        const int src = __builtin_ctzll(b);
        lane_heap_push_root(hd, hi, lane, k, lane_value(v[u], src), static_cast<uint32_t>(r0 + 64 * u + src));
        top = lane_value(hd, 0);
        b &= b - 1;
        b &= __ballot(v[u] < top);
      }
    }
#pragma unroll
    for (int u = 0; u < kFewLoads; ++u) v[u] = w[u];
  }
  lane_heap_store(hd, hi, lane, k, out_idx + qi * k, out_dist + qi * k, out_count + qi);
}

template <typename T, int M>
int run_few(const sc_index* index, const T* d_queries, int64_t q, int k, int64_t* d_idx, double* d_dist,
            uint32_t* d_count, hipStream_t s) {
  const int64_t n = static_cast<int64_t>(index->n), npad = (n + kFewChunk - 1) / kFewChunk * kFewChunk;
  const int ld = static_cast<int>(index->ld);
  DevBuf dist;
  SC_HIP(dist.alloc(sizeof(double) * q * npad, s));
  {
    ProfScope ps("knn_scan", s);
    hipLaunchKernelGGL((few_sums_kernel<T, M>),
                       dim3(static_cast<unsigned>(npad / kFewThreads), static_cast<unsigned>(q)),
                       dim3(kFewThreads), sizeof(T) * ld, s, static_cast<const T*>(index->rows), n, npad, ld,
                       d_queries, dist.as<double>());
    SC_HIP(hipGetLastError());
  }
  ProfScope ps("knn_replay", s);
  hipLaunchKernelGGL(few_replay_kernel, dim3(static_cast<unsigned>(q)), dim3(64), 0, s, dist.as<double>(), npad,
                     k, d_idx, d_dist, d_count);
  SC_HIP(hipGetLastError());
  return SC_OK;
}

}  // namespace

// Measured from host arrays, this form against the general one (f64, k = 5;
// us): 1 query x 10,000 x 32: 48 and 83; x 65,536 x 32: 80 and 105; x 131,072
// x 32: 133 and 131, for the replay walks every distance; 64 queries x 32,768
// x 32 (6.7e7 values): 98 and 117; x 65,536 x 32 (1.3e8): 154 and 124, for
// each query reads all rows; 1,024 queries x 1,000 x 32: 87 and 116; 4,096: 217
// and 212.  Manhattan's general form is slower yet (64 x 1,000 x 32: 42 and 176).
constexpr size_t kFewRows = 65536, kFewQueries = 1024, kFewWork = 80000000;
bool knn_few_applies(const sc_index* index, size_t q, size_t k, sc_metric metric) {
  return k <= 64 && (metric == SC_EUCLIDIAN || metric == SC_MANHATTAN) && q <= kFewQueries && index->n <= kFewRows &&
         q * index->n * index->ld <= kFewWork && index->ld * elem_size(index->dtype) <= 32768;
}

int knn_few_device(const sc_index* index, const void* d_queries, size_t q, size_t k, sc_metric metric,
                   int64_t* d_idx, double* d_dist, uint32_t* d_count, hipStream_t s, sc_stats* stats) {
  const int64_t qn = static_cast<int64_t>(q);
  const int kk = static_cast<int>(k);
  int rc;
  if (index->dtype == SC_F64) {
    const double* qs = static_cast<const double*>(d_queries);
    rc = metric == SC_EUCLIDIAN ? run_few<double, kEuclid>(index, qs, qn, kk, d_idx, d_dist, d_count, s)
                                : run_few<double, kManhattan>(index, qs, qn, kk, d_idx, d_dist, d_count, s);
  } else {
    const float* qs = static_cast<const float*>(d_queries);
    rc = metric == SC_EUCLIDIAN ? run_few<float, kEuclid>(index, qs, qn, kk, d_idx, d_dist, d_count, s)
                                : run_few<float, kManhattan>(index, qs, qn, kk, d_idx, d_dist, d_count, s);
  }
  if (rc == SC_OK && stats) {
    stats->queries += q;
    stats->candidates += q * index->n;
  }
  return rc;
}

}  // namespace sc
