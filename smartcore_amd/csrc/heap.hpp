// The reference heap (HeapSelection, heap_select.rs) held across the lanes
// of one wavefront, shared by every replay kernel.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace sc {

__device__ __forceinline__ double lane_value(double v, int l) {
  const int lo = __builtin_amdgcn_readlane(static_cast<int>(__double_as_longlong(v)), l);
  const int hi = __builtin_amdgcn_readlane(static_cast<int>(__double_as_longlong(v) >> 32), l);
  return __longlong_as_double((static_cast<long long>(hi) << 32) |
                              static_cast<unsigned long long>(static_cast<uint32_t>(lo)));
}
__device__ __forceinline__ float lane_value(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// Lane j < k holds heap entry j (distance hd, row hi).  Replacing the root
// and sifting it down follows HeapSelection::sift_down
// (heap_select.rs:71-86: the children of kk are 2kk and 2kk + 1; stop on
// Equal or Greater) with the node values read by readlane and the swap done
// by a select in every lane, so an insertion costs a few instructions per
// level and no memory traffic.
__device__ __forceinline__ void lane_heap_push_root(double& hd, uint32_t& hi, int lane, int k,
                                                    double d, uint32_t row) {
  if (lane == 0) {
    hd = d;
    hi = row;
  }
  const int n = k - 1;
  int kk = 0;
  const double vk = d;
  while (2 * kk <= n) {
    int j = 2 * kk;
    double vj = lane_value(hd, j);
    if (j < n) {
      const double vj1 = lane_value(hd, j + 1);
      if (vj < vj1) {
        j += 1;
        vj = vj1;
      }
    }
    if (vk == vj || vk > vj) break;
    const uint32_t ij = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(hi), j));
    const uint32_t ik = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(hi), kk));
    if (lane == kk) {
      hd = vj;
      hi = ij;
    } else if (lane == j) {
      hd = vk;
      hi = ik;
    }
    kk = j;
  }
}

// The heap's final state as LinearKNNSearch::find returns it
// (linear_search.rs:79-83): heap-array order without the empty slots, padded
// with -1 / NaN.
__device__ __forceinline__ void lane_heap_store(double hd, uint32_t hi, int lane, int k,
                                                int64_t* __restrict__ out_idx,
                                                double* __restrict__ out_dist,
                                                uint32_t* __restrict__ out_count) {
  const bool full = lane < k && hi != 0xffffffffu;
  const uint64_t fm = __ballot(full);
  const int c = __popcll(fm);
  if (full) {
    const int pos = __popcll(fm & ((uint64_t(1) << lane) - 1));
    out_idx[pos] = static_cast<int64_t>(hi);
    out_dist[pos] = hd;
  }
  if (lane >= c && lane < k) {
    out_idx[lane] = -1;
    out_dist[lane] = NAN;
  }
  if (lane == 0) *out_count = static_cast<uint32_t>(c);
}

}  // namespace sc
