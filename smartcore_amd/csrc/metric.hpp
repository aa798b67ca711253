// Per-element distance terms in the reference's exact arithmetic.
//
// Each term is one summand of the left fold the reference computes; the
// caller accumulates `s = s + term` in f64 with separate roundings (the
// library is compiled with -ffp-contract=off so no FMA is formed).
#pragma once

#include <hip/hip_runtime.h>

namespace sc {

enum MetricId : int { kEuclid = 0, kManhattan = 1, kMinkowski = 2 };

template <typename T, int M>
struct Term;

// euclidian.rs:57-62, T = f64: r = a - b; (r * r) as f64
template <>
struct Term<double, kEuclid> {
  static __device__ __forceinline__ double f(double a, double b, double) {
    double r = a - b;
    return r * r;
  }
};
// euclidian.rs:57-62, T = f32: r and r * r rounded in f32, then widened
template <>
struct Term<float, kEuclid> {
  static __device__ __forceinline__ double f(float a, float b, double) {
    float r = a - b;
    float r2 = r * r;
    return static_cast<double>(r2);
  }
};
// manhattan.rs:56-59: (a - b).to_f64().abs()
template <>
struct Term<double, kManhattan> {
  static __device__ __forceinline__ double f(double a, double b, double) { return fabs(a - b); }
};
template <>
struct Term<float, kManhattan> {
  static __device__ __forceinline__ double f(float a, float b, double) {
    float r = a - b;
    return fabs(static_cast<double>(r));
  }
};
// minkowski.rs:61-64: (a - b).to_f64().abs().powf(p)
template <>
struct Term<double, kMinkowski> {
  static __device__ __forceinline__ double f(double a, double b, double p) {
    return pow(fabs(a - b), p);
  }
};
template <>
struct Term<float, kMinkowski> {
  static __device__ __forceinline__ double f(float a, float b, double p) {
    float r = a - b;
    return pow(fabs(static_cast<double>(r)), p);
  }
};

// The reference's sum of one (query, row) pair (p-free metrics): terms in dimension order,
// 16 values of both requested before they are folded (rows are padded to
// multiples of 16 values).
template <typename T, int M>
__device__ __forceinline__ double exact_sum(const T* __restrict__ x, const T* __restrict__ y, int ld) {
  constexpr int PV = 16 / sizeof(T);
  typedef T Piece __attribute__((ext_vector_type(PV)));
  const Piece* xp = reinterpret_cast<const Piece*>(x);
  const Piece* yp = reinterpret_cast<const Piece*>(y);
  double s = 0.0;
  for (int j = 0; j < ld / PV; j += 16 / PV) {
    Piece xv[16 / PV], yv[16 / PV];
#pragma unroll
    for (int c = 0; c < 16 / PV; ++c) {
      xv[c] = xp[j + c];
      yv[c] = yp[j + c];
    }
#pragma unroll
    for (int c = 0; c < 16 / PV; ++c)
#pragma unroll
      for (int w = 0; w < PV; ++w) s = s + Term<T, M>::f(xv[c][w], yv[c][w], 0.0);
  }
  return s;
}

// The sums of up to 64 (query, row) pairs by one wavefront, lane = row.  A
// lane that reads its own row asks for 64 lines per load, and the address
// unit takes them one by one; here four lanes read 64 bytes of a row, so a
// load touches sixteen lines, and the rows go through an LDS tile from which
// each lane folds its own in dimension order.  x: the query row, in LDS.  All
// lanes take part (row: any valid row for the idle ones).
constexpr int kSumTileStride = 64 + 16;  // bytes of a row's 64 in the tile
constexpr int kSumTileBytes = 64 * kSumTileStride;
template <typename T, int M>
__device__ __forceinline__ double wave_exact_sums(const T* x, const T* __restrict__ rows,
                                                  uint32_t row, int ld, unsigned char* tile) {
  constexpr int PV = 16 / sizeof(T);
  constexpr int CW = 64 / sizeof(T);  // values of a chunk (ld is a multiple)
  typedef T Piece __attribute__((ext_vector_type(PV)));
  const int lane = threadIdx.x & 63;
  const T* src[4];
#pragma unroll
  for (int p = 0; p < 4; ++p)
    src[p] = rows + static_cast<int64_t>(__shfl(row, 16 * p + (lane >> 2))) * ld + (lane & 3) * PV;
  Piece v[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) v[p] = *reinterpret_cast<const Piece*>(src[p]);
  double s = 0.0;
  for (int c0 = 0; c0 < ld; c0 += CW) {
#pragma unroll
    for (int p = 0; p < 4; ++p)
      *reinterpret_cast<Piece*>(tile + (16 * p + (lane >> 2)) * kSumTileStride + 16 * (lane & 3)) = v[p];
    if (c0 + CW < ld) {  // the next chunk is on its way while this one is folded
#pragma unroll
      for (int p = 0; p < 4; ++p) v[p] = *reinterpret_cast<const Piece*>(src[p] + c0 + CW);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    Piece y[4];
#pragma unroll
    for (int p = 0; p < 4; ++p)
      y[p] = *reinterpret_cast<const Piece*>(tile + lane * kSumTileStride + 16 * p);
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int w = 0; w < PV; ++w) s = s + Term<T, M>::f(x[c0 + p * PV + w], y[p][w], 0.0);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  return s;
}

// Distance from the folded sum: euclidian.rs:71 sqrt, manhattan identity,
// minkowski.rs:66 powf(1/p).  The selection kernels filter on the sum, which
// is valid because each finaliser is monotone non-decreasing.
template <int M>
__device__ __forceinline__ double finalize(double s, double p) {
  if constexpr (M == kEuclid) {
    return __builtin_sqrt(s);
  } else if constexpr (M == kManhattan) {
    return s;
  } else {
    return pow(s, 1.0 / p);
  }
}

}  // namespace sc
