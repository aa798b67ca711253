// FP64 MFMA tile sweep shared by the Euclidian searches.
//
// A 256-thread workgroup sweeps 128-row tiles of the index against 128
// queries.  Wave w owns queries 32 w .. 32 w + 31 against all 128 rows, as
// 8 x 2 v_mfma_f64_16x16x4_f64 accumulators (128 VGPRs): a K step of four
// dimensions costs 10 LDS reads for 16 MFMAs, and because a query's rows
// never leave its wavefront, results are filtered and appended in row order
// without a barrier (a 2 x 2 arrangement of 64 x 64 needs 8 reads, but two
// barriers per tile to order a query's rows across two wavefronts: 4,096
// queries x 200,000 x 64 took 2.91 ms with it and 2.56 ms without, 5,000 x
// 100,000 x 16 within a radius 0.91 and 0.84).  What it needs most is the
// matrix pipe (64 cycles per MFMA and SIMD): the vector form needs three FP64
// instructions per element (subtract, multiply, add) where the MFMA needs one
// fused multiply-add.  It reaches 64 % of a large matrix product's rate at 64
// dimensions and 76 % at 100: a barrier per 16 dimensions, and at a tile's end
// 64 FP64 compares per lane beside an idle matrix pipe, whatever the rows' length.
// Dimension chunks of 16 go through two LDS buffers: chunk c + 1 is stored
// and chunk c + 2 requested while chunk c's MFMAs run, with one barrier per
// chunk; the chunk stream runs on across tiles, so a tile's first chunk is
// as early as any other.  Queries of one chunk are staged once.  f32 rows
// are widened (exactly) when they are stored to LDS.
//
// The accumulators start at y2m, a lower bound of the row's ||y||^2, and the
// queries are staged as -2x, so a tile ends with acc = y2m - 2 x.y.
//
// Bound.  With D = ||x - y||^2 exactly, u = 2^-53 and any order of the
// accumulation, the MFMA chain's error is at most 2 ld u (x2 + y2) for the
// products' sum plus the same for the running sum that contains y2m, and the
// norms carry (ld + 1) u each.  norm_gap(ld) = g = (4 ld + 32) 2^-52 is above
// all of it, so with x2m = (1 - g) x2 and y2m = (1 - g) y2
//   L = x2m + acc <= D <= L + 2.5 g (x2m + y2m).
// The reference's sum S (euclidian.rs:57-62) is within sum_eps of D in
// relative terms and sum_tiny absolutely (f32 squares may underflow), so
//   S < T  implies  acc < T (1 + 3 eps) + 2 tiny - x2m.
// Rows with a non-finite value never enter the reference heap or pass a
// radius test (their S is inf or NaN); they carry y2m = +inf and are left
// out.  Rows whose squared norm reaches kNorm64Limit carry NaN: comparisons
// are written so that NaN is always a candidate, and exact arithmetic
// decides.
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"
#include "metric.hpp"

namespace sc {

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int kMQ = 128;       // queries per workgroup tile
constexpr int kMR = 128;       // rows per tile
constexpr int kMD = 16;        // dimensions per chunk
constexpr int kMT = 256;       // threads
// LDS row stride of a chunk: 16 values + 2, so the 16 rows x 4 dimensions a
// wave reads with one ds_read_b64 fall on every bank exactly twice
constexpr int kMStride = kMD + 2;
constexpr double kNorm64Limit = 1e290;

inline double norm_gap(int ld) { return (4.0 * ld + 32.0) * 2.220446049250313e-16; }
template <typename T>
inline double sum_eps(int ld) {
  // f64: three roundings per term and ld adds; f32: two f32 roundings of
  // the difference (squared) and one of the square, then the f64 fold
  return sizeof(T) == 8 ? (ld + 8.0) * 2.220446049250313e-16
                        : 2.384185791015625e-07 + (ld + 8.0) * 2.220446049250313e-16;
}
template <typename T>
inline double sum_tiny(int ld) {
  return sizeof(T) == 8 ? 1e-300 : ld * 2.802596928649634e-45;
}
// Above this a sum may overflow in the reference's own type.
template <typename T>
inline double sum_limit() {
  return sizeof(T) == 8 ? 1e300 : 1e38;
}
// The bound's constants as the kernels take them.
struct Bound64 {
  double gap25;   // 2.5 g
  double up;      // 1 + 3 eps
  double tiny;    // 2 tiny
  double limit;
};
template <typename T>
inline Bound64 bound64(int ld) {
  return Bound64{2.5 * norm_gap(ld), 1.0 + 3.0 * sum_eps<T>(ld), 2.0 * sum_tiny<T>(ld),
                 sum_limit<T>()};
}
// The accumulator threshold that every row with S < t is below.
__device__ __forceinline__ double acc_threshold(const Bound64& b, double t, double x2m) {
  return t < INFINITY ? t * b.up + b.tiny - x2m : INFINITY;
}
// An upper bound on S of a pair whose lower bound on D is L.
__device__ __forceinline__ double sum_upper(const Bound64& b, double L, double norms) {
  const double u = (L + b.gap25 * norms) * b.up + b.tiny;
  return u < b.limit ? u : INFINITY;  // NaN too
}

struct MSmem {
  double R[2][kMR][kMStride];
  double Q[2][kMQ][kMStride];
  // y2m by tile modulo 4: a wavefront may still read a tile's while the
  // others, at most one barrier ahead, store the next but one's
  double y2[4][kMR];
};

// Where a lane's accumulators lie: acc[i][j][v] is row row_of(i, v), query
// query_of(j) of the tile.  The four lanes of a query's column hold four
// consecutive rows.
struct MLane {
  int lane, wave, lr, lg;
  __device__ __forceinline__ MLane() {
    lane = threadIdx.x & 63;
    wave = threadIdx.x >> 6;
    lr = lane & 15;
    lg = lane >> 4;
  }
  __device__ __forceinline__ int row_of(int i, int v) const { return 16 * i + 4 * v + lg; }
  __device__ __forceinline__ int query_of(int j) const { return wave * 32 + 16 * j + lr; }
  // the lanes of this lane's column
  __device__ __forceinline__ uint64_t column() const { return uint64_t(0x0001000100010001) << lr; }
  __device__ __forceinline__ uint64_t below() const { return (uint64_t(1) << lane) - 1; }
};
typedef f64x4 MAcc[8][2];

// Sweeps tiles at(tb) .. at(te - 1) (row = row0 + 128 tile) against queries
// q0 .. q0 + 127; epi(t, acc, slot) runs at the end of tile at(t), without a
// barrier of its own (sm.y2[slot] holds the tile's y2m).  Out-of-range rows and
// queries are read clamped: y2m carries +inf past the last row.  SWAP: the
// accumulators hold (query, row) transposed -- acc[i][j][v] of a lane is row
// 16 i + lr, query 32 wave + 16 j + 4 v + lg -- and start at zero.
template <typename T, bool SWAP, typename Epi, typename At>
__device__ __forceinline__ void mfma64_sweep(MSmem& sm, const T* __restrict__ rows, int64_t n,
                                             int ld, int d, const double* __restrict__ y2m,
                                             const T* __restrict__ queries, int64_t q, int64_t q0,
                                             int64_t row0, int64_t tb, int64_t te, Epi epi, At at) {
  constexpr int PV = 16 / sizeof(T);            // values per 16-byte piece
  constexpr int PR = kMD / PV;                  // pieces per row of a chunk
  constexpr int NP = kMR * PR / kMT;            // pieces per thread (rows and queries each)
  typedef T Piece __attribute__((ext_vector_type(PV)));
  const int tid = threadIdx.x;
  const MLane ml;
  const int nch = d > kMD ? (d + kMD - 1) / kMD : 1;
  const int64_t total = (te - tb) * nch;
  if (total <= 0) return;

  // this thread's pieces: row (or query) pr + p * (kMT / PR), values pc ..
  const int pr = tid / PR, pc = (tid % PR) * PV;
  // (32-bit offsets from the query tile's first row)
  const T* qbase = queries + q0 * ld;
  const int qleft = static_cast<int>(min<int64_t>(kMQ, q - q0)) - 1;
  Piece vr[NP], vq[NP];
  double vy = 0.0;
  int64_t lt = tb;  // load cursor: tile and chunk
  int lk = 0;
  auto gload_q = [&]() {
    const T* cbase = qbase + lk * kMD;
#pragma unroll
    for (int p = 0; p < NP; ++p)
      vq[p] = *reinterpret_cast<const Piece*>(cbase + min(pr + p * (kMT / PR), qleft) * ld + pc);
  };
  auto gload = [&]() {
    const int64_t t0 = row0 + at(lt) * kMR;
    const T* rbase = rows + t0 * ld + lk * kMD;
    const int left = static_cast<int>(min<int64_t>(kMR, n - t0)) - 1;
#pragma unroll
    for (int p = 0; p < NP; ++p)
      vr[p] = *reinterpret_cast<const Piece*>(rbase + min(pr + p * (kMT / PR), left) * ld + pc);
    if (nch > 1) gload_q();
    if (lk == 0 && tid < kMR) vy = y2m[t0 + tid];
  };
  auto swrite_q = [&](int buf) {
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int c = 0; c < PV; ++c)
        sm.Q[buf][pr + p * (kMT / PR)][pc + c] = -2.0 * static_cast<double>(vq[p][c]);
  };
  auto swrite = [&](int buf) {
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int c = 0; c < PV; ++c)
        sm.R[buf][pr + p * (kMT / PR)][pc + c] = static_cast<double>(vr[p][c]);
    if (nch > 1) swrite_q(buf);
    if (lk == 0 && tid < kMR) sm.y2[(lt - tb) & 3][tid] = vy;
  };
  auto advance = [&]() {
    if (++lk == nch) {
      lk = 0;
      ++lt;
    }
  };
  if (nch == 1) {  // the queries' only chunk: staged for the whole sweep
    gload_q();
    swrite_q(0);
  }
  gload();
  swrite(0);
  advance();
  if (total > 1) gload();
  __syncthreads();

  MAcc acc;
  int kc = 0;
  int64_t t = tb;
  for (int64_t c = 0; c < total; ++c) {
    const int buf = static_cast<int>(c & 1);
    const int qbuf = nch > 1 ? buf : 0;
    const int par = static_cast<int>((t - tb) & 3);
    if (c + 1 < total) {
      swrite(buf ^ 1);
      advance();
      if (c + 2 < total) gload();
    }
    if (kc == 0) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        f64x4 y = {0.0, 0.0, 0.0, 0.0};
        if (!SWAP) {
#pragma unroll
          for (int v = 0; v < 4; ++v) y[v] = sm.y2[par][ml.row_of(i, v)];
        }
        acc[i][0] = y;
        acc[i][1] = y;
      }
    }
    // K step s covers dimensions 4s .. 4s + 3 of the chunk; the last chunk
    // stops at the row's true dimension (the padding is zeros)
    const int steps = min(4, (d - kc * kMD + 3) / 4);
#pragma unroll 1
    for (int s = 0; s < steps; ++s) {
      double a[8], b[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) b[j] = sm.Q[qbuf][ml.wave * 32 + 16 * j + ml.lr][4 * s + ml.lg];
#pragma unroll
      for (int i = 0; i < 8; ++i) a[i] = sm.R[buf][16 * i + ml.lr][4 * s + ml.lg];
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = SWAP ? __builtin_amdgcn_mfma_f64_16x16x4f64(b[j], a[i], acc[i][j], 0, 0, 0)
                           : __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
    if (++kc == nch) {
      epi(t, acc, par);
      kc = 0;
      ++t;
    }
  }
}

// The tiles tb .. te - 1 themselves.
template <typename T, bool SWAP, typename Epi>
__device__ __forceinline__ void mfma64_sweep(MSmem& sm, const T* __restrict__ rows, int64_t n,
                                             int ld, int d, const double* __restrict__ y2m,
                                             const T* __restrict__ queries, int64_t q, int64_t q0,
                                             int64_t row0, int64_t tb, int64_t te, Epi epi) {
  mfma64_sweep<T, SWAP>(sm, rows, n, ld, d, y2m, queries, q, q0, row0, tb, te, epi,
                        [](int64_t t) { return t; });
}

// Calls f(i, j, v, row, hit, mask) for every accumulator register of the
// wavefront that holds values below their query's threshold th[j] (-inf: a
// query that takes no part), rows ascending for each query; hit: this lane
// is one of the lanes in mask.  Rows that y2 leaves out are dropped.  The
// first test of a query block is one compare per register, or-ed in scalar
// registers.
template <typename F>
__device__ __forceinline__ void tile_hits(const MLane& ml, const MAcc& acc, const double (&th)[2],
                                          const double* y2, F f) {
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    uint64_t some = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) some |= __ballot(!(acc[i][j][v] >= th[j]));
    if (some == 0) continue;  // the whole wavefront
    // compared anew: 32 kept compare masks would not fit the scalar registers
    double t = th[j];
    asm volatile("" : "+v"(t));
    const bool part = !(t == -INFINITY);
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        bool hit = !(acc[i][j][v] >= t);
        if (__ballot(hit) == 0) continue;
        const int rl = ml.row_of(i, v);
        hit = hit && part && y2[rl] != INFINITY;
        const uint64_t m = __ballot(hit);
        if (m) f(i, j, v, rl, hit, m);
      }
  }
}

// y2m of every row of an index (kMR rows of padding past the last, +inf),
// built once per index on the stream of the first call, which does not wait
// for it.  Until it is complete, calls on other streams build their own into
// `local` (waiting for it would put them behind all that the first stream has
// queued), and so do those on a capturing stream, where nothing may be kept or
// waited for.
int ensure_norms64(sc_index* ix, DevBuf& local, const double** y2m, hipStream_t s);
// The same for a call's queries (no padding).  Queries with a finite but too
// large norm are appended to list (their x2m is +inf, like that of the
// non-finite ones).
template <typename T>
int query_norms64(const T* queries, int64_t q, int ld, double* x2m, uint32_t* list,
                  uint32_t* list_n, hipStream_t s);

}  // namespace sc
