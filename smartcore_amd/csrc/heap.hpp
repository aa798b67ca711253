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
__device__ __forceinline__ uint32_t lane_value(uint32_t v, int l) {
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), l));
}
__device__ __forceinline__ float lane_value(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// The value of lane ^ 1 (quad permutation 1, 0, 3, 2).
__device__ __forceinline__ double lane_xor1(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(static_cast<int>(__double_as_longlong(v)), 0xB1, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(static_cast<int>(__double_as_longlong(v) >> 32), 0xB1, 0xf, 0xf, true);
  return __longlong_as_double((static_cast<long long>(hi) << 32) |
                              static_cast<unsigned long long>(static_cast<uint32_t>(lo)));
}

// Lane j < k holds heap entry j (distance hd, row hi).  Replaces the root by
// (d, row), d below the root's distance, and sifts it down as
// HeapSelection::sift_down does (heap_select.rs:71-86: the children of kk are
// 2kk and 2kk + 1, so the root's child is 1; the larger child, the first of
// equals, is taken; stop on Equal or Greater).  The path does not depend on
// the new value, only where it stops does, so all levels are done at once:
// every lane tells whether it is the larger of its pair, a lane is on the
// path when it and all its ancestors are, and the entries of the path above
// d move up one place.  One neighbour exchange, one ballot and one shuffle,
// whatever the depth: following the path with one readlane after another took
// about 1,000 cycles at k = 20, and the replay of 240 entrants a quarter of a
// millisecond.
__device__ __forceinline__ void lane_heap_push_root(double& hd, uint32_t& hi, int lane, int k,
                                                    double d, uint32_t row) {
  const int n = k - 1;
  const double sib = lane_xor1(hd);
  const bool larger = (lane & 1) ? sib < hd : !(lane < n && hd < sib);
  const uint64_t c = __ballot(lane >= 2 && lane <= n && larger) | 3u;
  // on the path: bits lane, lane >> 1, lane >> 2, ... (bit 0 is set)
  const uint32_t clo = static_cast<uint32_t>(c), chi = static_cast<uint32_t>(c >> 32);
  uint32_t on = lane < 32 ? clo >> lane : chi >> (lane - 32);
  on &= clo >> (lane >> 1);
  on &= clo >> (lane >> 2);
  on &= clo >> (lane >> 3);
  on &= clo >> (lane >> 4);
  on &= clo >> (lane >> 5);
  // the larger child and its entry
  const int first = 2 * lane;
  const bool parent = lane == 0 ? n >= 1 : first <= n;
  const uint32_t odd = lane < 16 ? (clo >> (first + 1)) & 1u : (chi >> ((first + 1) & 31)) & 1u;
  const int child = lane == 0 ? 1 : first + static_cast<int>(odd);
  const double cd = __shfl(hd, child & 63);
  const uint32_t ci = __shfl(hi, child & 63);
  if (lane == 0 || ((on & 1u) && lane <= n && hd > d)) {
    const bool up = parent && cd > d;
    hd = up ? cd : d;
    hi = up ? ci : row;
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
