// SC_MIXED Manhattan kNN on 16-bit codes (f32 rows).  The index's values are coded as
// c = clamp(rint((v - lo) / h), 0, 65535) with h a power of two and lo a
// multiple of h, so deq(c) = lo + c h is exact in f64.  Per row the code
// error er >= sum_i |y_i - deq(c_i)| / h (an integer, rounded up); per query
// eq >= sum_i |x_i - deq(c_i)| / h (f64, rounded up; clamping included).
// With D = sum_i |x_i - y_i| and sad = sum_i |cx_i - cy_i| (v_sad_u16, two
// dimensions per instruction, exact in u32), the triangle inequality gives
//   h (sad - eq - er) <= D <= h (sad + eq + er).
// The reference sum S = f64 fold of |fl32(x_i - y_i)| (manhattan.rs:56-59)
// lies in [(1 - eps) D, (1 + eps) D], eps = 2^-24 + (d + 1) 2^-52 (one f32
// rounding per term, at most d f64 roundings of the fold), so
//   L = (1 - eps) h (sad - eq - er) <= S <= U = (1 + eps) h (sad + eq + er).
// The scan keeps per query the k smallest V = sad + er (the k smallest U)
// and stores every row with L below the running k-th U, i.e. with
//   W = sad - er < rho (V_k + eq) + eq,  rho >= (1 + eps) / (1 - eps),
// tested in integers against the right side rounded up.  Padding dimensions
// code to 0 on both sides and add nothing.
//
//   dense    W of every query against the first rows, written out; select0
//            walks it in row order for the prefix's candidates and the first
//            k-th V.
//   scan     The rest in levels (knn_lists.hpp).  A workgroup sweeps 128-row
//            tiles against 128 queries; a wavefront owns 32 queries against
//            all 128 rows, each lane an 8 x 8 register tile, so that eight
//            LDS words feed 64 v_sad_u16 (58 % of the 35 T lane
//            instructions/s of this card at 96 dimensions: each dword's LDS
//            reads are waited for before its sads, and the tile spills), and a
//            query's hits are appended in row order without a barrier.  Up
//            to 32 queries, the four wavefronts take four pieces of the rows
//            against the same queries instead, and the rows' bytes bound it.
//   finish   The reference sums of the candidates and the heap replay.
// 1,024 queries x 1,000,000 x 96, k = 20: 2.4 ms (6.9 with 32 x 128 tiles
// of 4 x 4 per lane, where LDS reads bound the scan and a thread per query
// kept its k best for every row).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

#include "common.hpp"
#include "knn_lists.hpp"
#include "metric.hpp"

namespace sc {

// from knn_exact.hip
int launch_serial_manhattan_f32(const sc_index* index, const float* d_queries, int k,
                                const uint32_t* list, const uint32_t* list_n, int64_t* d_idx,
                                double* d_dist, uint32_t* d_count, hipStream_t stream);

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr double kQ16Limit = 1e30;

// thr = ceil(rho (vk + eq) + eq) with every operation rounded up; "no
// threshold" (fewer than k rows seen, or a query outside the domain) is
// INT_MAX, which every W is below.
__device__ __forceinline__ int q16_threshold(uint32_t vk, double eq, double rho) {
  if (vk == 0xffffffffu || !(eq < INFINITY)) return 0x7fffffff;
  const double r = __ocml_add_rtp_f64(
      __ocml_mul_rtp_f64(__ocml_add_rtp_f64(static_cast<double>(vk), eq), rho), eq);
  const double c = ceil(r);
  return c >= 2147483647.0 ? 0x7fffffff : static_cast<int>(c);
}

// Range of the index's values (first d of each row): per block min, max,
// sum |v| and a flag for values outside the form's domain.
__global__ void q16_range_kernel(const float* __restrict__ rows, int64_t n, int d, int ld,
                                 double* __restrict__ part) {
  __shared__ double smin[256], smax[256], ssum[256], sbad[256];
  double mn = INFINITY, mx = -INFINITY, sm = 0.0, bad = 0.0;
  // sixteen lanes per row
  const int sub = threadIdx.x & 15;
  for (int64_t r = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) >> 4; r < n;
       r += (static_cast<int64_t>(gridDim.x) * blockDim.x) >> 4) {
    for (int j = sub; j < d; j += 16) {
      const double v = rows[r * ld + j];
      if (!(fabs(v) <= kQ16Limit)) {
        bad = 1.0;
        continue;
      }
      mn = fmin(mn, v);
      mx = fmax(mx, v);
      sm += fabs(v);
    }
  }
  const int t = threadIdx.x;
  smin[t] = mn;
  smax[t] = mx;
  ssum[t] = sm;
  sbad[t] = bad;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (t < s) {
      smin[t] = fmin(smin[t], smin[t + s]);
      smax[t] = fmax(smax[t], smax[t + s]);
      ssum[t] += ssum[t + s];
      sbad[t] = fmax(sbad[t], sbad[t + s]);
    }
    __syncthreads();
  }
  if (t == 0) {
    part[4 * blockIdx.x + 0] = smin[0];
    part[4 * blockIdx.x + 1] = smax[0];
    part[4 * blockIdx.x + 2] = ssum[0];
    part[4 * blockIdx.x + 3] = sbad[0];
  }
}

// Codes of one vector's value (f64 arithmetic; deq(c) = lo + c h exact) and
// the absolute code error.
__device__ __forceinline__ uint32_t q16_code(float v, double lo, double h, double inv_h,
                                             double* err) {
  double c = rint((static_cast<double>(v) - lo) * inv_h);
  c = fmin(fmax(c, 0.0), 65535.0);
  *err += fabs(static_cast<double>(v) - (lo + c * h));
  return static_cast<uint32_t>(c);
}

// Codes of one vector by eight lanes (dimension pairs in dwords, padding
// dimensions 0); returns the code error in units of h and whether every
// value is in the form's domain.
__device__ __forceinline__ double q16_vector(const float* __restrict__ r, int d, int ld, double lo,
                                             double h, double inv_h, int sub,
                                             uint32_t* __restrict__ o, bool* ok) {
  double err = 0.0;
  bool in = true;
  for (int w = sub; w < ld / 2; w += 8) {
    const float2 v = *reinterpret_cast<const float2*>(r + 2 * w);
    uint32_t c0 = 0u, c1 = 0u;
    if (2 * w < d) {
      c0 = q16_code(v.x, lo, h, inv_h, &err);
      in = in && fabsf(v.x) <= static_cast<float>(kQ16Limit);
    }
    if (2 * w + 1 < d) {
      c1 = q16_code(v.y, lo, h, inv_h, &err);
      in = in && fabsf(v.y) <= static_cast<float>(kQ16Limit);
    }
    o[w] = c0 | (c1 << 16);
  }
#pragma unroll
  for (int s = 4; s >= 1; s >>= 1) {
    err += __shfl_xor(err, s, 8);
    in = (__shfl_xor(static_cast<int>(in), s, 8) != 0) && in;
  }
  *ok = in;
  return err * inv_h;
}

// Rows: codes and er (0 for the padding rows).
__global__ void q16_rows_kernel(const float* __restrict__ rows, int64_t n, int64_t npad, int d,
                                int ld, double lo, double h, uint32_t* __restrict__ codes,
                                uint32_t* __restrict__ er) {
  const int sub = threadIdx.x & 7;
  for (int64_t i = lane_row(8); i < npad; i += lane_row_step(8)) {  // eight lanes together
    uint32_t e = 0u;
    if (i < n) {
      bool ok;
      const double err = q16_vector(rows + i * ld, d, ld, lo, h, 1.0 / h, sub, codes + i * (ld / 2), &ok);
      // err carries at most two roundings per term (the difference, the add):
      // scale it up by more than that, then round up to an integer
      e = static_cast<uint32_t>(ceil(err * (1.0 + (2.0 * d + 4.0) * 2.220446049250313e-16)));
    }
    if (sub == 0) er[i] = e;
  }
}

// Queries: codes (clamped) and eq; a query with a value outside the domain
// gets eq = +inf and is listed for the serial kernel.
__global__ void q16_queries_kernel(const float* __restrict__ qs, int64_t q, int d, int ld,
                                   double lo, double h, uint32_t* __restrict__ codes,
                                   double* __restrict__ eq, uint32_t* __restrict__ list,
                                   uint32_t* __restrict__ list_n) {
  const int sub = threadIdx.x & 7;
  for (int64_t i = lane_row(8); i < q; i += lane_row_step(8)) {
    bool ok;
    const double err = q16_vector(qs + i * ld, d, ld, lo, h, 1.0 / h, sub, codes + i * (ld / 2), &ok);
    if (sub != 0) continue;
    eq[i] = ok ? __ocml_mul_rtp_f64(err, 1.0 + (2.0 * d + 4.0) * 2.220446049250313e-16) : INFINITY;
    if (!ok) list[atomicAdd(list_n, 1u)] = static_cast<uint32_t>(i);
  }
}


// One chunk of codes: kSadChunk dwords (two dimensions each) of the tile's
// rows and queries, transposed so that a lane reads its four consecutive rows
// (or queries) of a dword with one 16-byte load.  QW: wavefronts along the
// queries (4: one row stream of 128 x 128 tiles; 1: four row streams against
// the same 32 queries).
constexpr int kSadChunk = 8;
constexpr int kSadThreads = 256;
template <int QW>
struct SadSmem {
  static constexpr int RW = 4 / QW;
  uint32_t R[2][kSadChunk][RW * kListTile + 4];
  uint32_t Q[2][kSadChunk][QW * 32 + 4];
};

// Where a lane's accumulators lie: acc[i][4 h + r] is query query_of(i) of
// its wavefront's 32, row row_of(h, r) of its stream's tile.
struct SadLane {
  int lane, wave, tr, g;
  __device__ __forceinline__ SadLane() {
    lane = threadIdx.x & 63;
    wave = threadIdx.x >> 6;
    tr = lane & 15;
    g = lane >> 4;
  }
  __device__ __forceinline__ int query_of(int i) const { return 8 * g + i; }
  __device__ __forceinline__ int row_of(int h, int r) const { return 64 * h + 4 * tr + r; }
  // the lanes that share this lane's queries
  __device__ __forceinline__ uint64_t peers() const { return uint64_t(0xffff) << (16 * g); }
  __device__ __forceinline__ uint64_t below() const { return (uint64_t(1) << lane) - 1; }
};
typedef uint32_t SadAcc[8][8];

// Sweeps nt tiles of each stream (stream w starts at row rb + w rstride)
// against queries q0 ..; epi(t, acc) at each tile's end, without a barrier of
// its own.  Rows and queries out of range are read clamped.
template <int QW, typename Epi>
__device__ __forceinline__ void sad_sweep(SadSmem<QW>& sm, const uint32_t* __restrict__ codes,
                                          int64_t n, int ldq, int ndw,
                                          const uint32_t* __restrict__ qcodes, int64_t q, int64_t q0,
                                          int64_t rb, int64_t rstride, int64_t nt, Epi epi) {
  constexpr int RW = SadSmem<QW>::RW;
  const int tid = threadIdx.x;
  const SadLane sl;
  const int nch = (ndw + kSadChunk - 1) / kSadChunk;
  const int64_t total = nt * nch;
  if (total <= 0) return;
  const int pr = tid >> 1, pc = 4 * (tid & 1);
  const bool has_q = QW == 4 || tid < 64;
  const int64_t qrow = min(q0 + pr, q - 1);
  u32x4 vr[RW], vq = {0u, 0u, 0u, 0u};
  int64_t lt = 0;
  int lk = 0;
  auto gload_q = [&]() {
    if (has_q) vq = *reinterpret_cast<const u32x4*>(qcodes + qrow * ldq + lk * kSadChunk + pc);
  };
  auto gload = [&]() {
#pragma unroll
    for (int w = 0; w < RW; ++w) {
      const int64_t r = min(rb + w * rstride + lt * kListTile + pr, n - 1);
      vr[w] = *reinterpret_cast<const u32x4*>(codes + r * ldq + lk * kSadChunk + pc);
    }
    if (nch > 1) gload_q();
  };
  auto swrite_q = [&](int buf) {
    if (has_q) {
#pragma unroll
      for (int c = 0; c < 4; ++c) sm.Q[buf][pc + c][pr] = vq[c];
    }
  };
  auto swrite = [&](int buf) {
#pragma unroll
    for (int w = 0; w < RW; ++w)
#pragma unroll
      for (int c = 0; c < 4; ++c) sm.R[buf][pc + c][w * kListTile + pr] = vr[w][c];
    if (nch > 1) swrite_q(buf);
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

  const int qoff = (QW == 4 ? sl.wave * 32 : 0) + 8 * sl.g;
  const int roff = (QW == 4 ? 0 : sl.wave * kListTile) + 4 * sl.tr;
  SadAcc acc;
  int kc = 0;
  int64_t t = 0;
  for (int64_t c = 0; c < total; ++c) {
    const int buf = static_cast<int>(c & 1);
    const int qbuf = nch > 1 ? buf : 0;
    if (c + 1 < total) {
      swrite(buf ^ 1);
      advance();
      if (c + 2 < total) gload();
    }
    if (kc == 0) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = 0u;
    }
    const int steps = min(kSadChunk, ndw - kc * kSadChunk);
    auto dword = [&](int s) {
      u32x4 a[2], b[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        a[h] = *reinterpret_cast<const u32x4*>(&sm.Q[qbuf][s][qoff + 4 * h]);
        b[h] = *reinterpret_cast<const u32x4*>(&sm.R[buf][s][roff + 64 * h]);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j)
          acc[i][j] = __builtin_amdgcn_sad_u16(a[i >> 2][i & 3], b[j >> 2][j & 3], acc[i][j]);
    };
    // (unrolled further, the reads are hoisted and the tile spills)
#pragma unroll 1
    for (int s = 0; s < steps; ++s) dword(s);
    __syncthreads();
    if (++kc == nch) {
      epi(t, acc);
      kc = 0;
      ++t;
    }
  }
}

// The lane's eight er values of a tile that starts at row r0 (er is padded
// to whole tiles).
__device__ __forceinline__ void tile_er(const SadLane& sl, const uint32_t* __restrict__ er, int64_t r0,
                                        int (&e)[8]) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const u32x4 v = *reinterpret_cast<const u32x4*>(er + r0 + sl.row_of(h, 0));
#pragma unroll
    for (int r = 0; r < 4; ++r) e[4 * h + r] = static_cast<int>(v[r]);
  }
}

// W of queries x the first `cols` rows (a multiple of kListTile, rows past
// the index INT_MAX), row-major by query.
__global__ __launch_bounds__(kSadThreads, 3) void l1q_dense_kernel(
    const uint32_t* __restrict__ codes, const uint32_t* __restrict__ er, int64_t n, int ldq, int ndw,
    const uint32_t* __restrict__ qcodes, int64_t q, int64_t cols, int* __restrict__ out) {
  __shared__ __align__(16) SadSmem<4> sm;
  const SadLane sl;
  const int64_t q0 = static_cast<int64_t>(blockIdx.x) * 128;
  const int64_t r0 = static_cast<int64_t>(blockIdx.y) * kListTile;
  sad_sweep<4>(sm, codes, n, ldq, ndw, qcodes, q, q0, r0, 0, 1, [&](int64_t, SadAcc& acc) {
    int e[8];
    tile_er(sl, er, r0, e);
    typedef int i32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int64_t qi = q0 + sl.wave * 32 + sl.query_of(i);
      if (qi >= q) continue;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        i32x4 w;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          w[r] = r0 + sl.row_of(h, r) < n ? static_cast<int>(acc[i][4 * h + r]) - e[4 * h + r]
                                          : 0x7fffffff;
        *reinterpret_cast<i32x4*>(out + qi * cols + r0 + sl.row_of(h, 0)) = w;
      }
    }
  });
}

__global__ __launch_bounds__(64 * kSelectWaves) void l1q_select_dense_kernel(
    const int* __restrict__ W, int64_t cols, const uint32_t* __restrict__ er,
    const double* __restrict__ eqv, int64_t q, int k, double rho, int cap,
    uint32_t* __restrict__ cand_idx, uint32_t* __restrict__ cand_count, uint32_t* __restrict__ seed) {
  const int lane = threadIdx.x & 63;
  const int64_t qi = static_cast<int64_t>(blockIdx.x) * kSelectWaves + (threadIdx.x >> 6);
  if (qi >= q) return;  // the whole wave
  const double eq = eqv[qi];
  KSmallest<uint32_t> ks;
  ks.clear();
  uint32_t cnt = 0;
  const int* w = W + qi * cols;
  if (eq < INFINITY) {
    int wv = w[lane];
    uint32_t ev = er[lane];
    int th = 0x7fffffff;
    // (past cap, the query's list is lost; what was seen stays a bound)
    for (int64_t c0 = 0; c0 < cols && cnt <= static_cast<uint32_t>(cap); c0 += 64) {
      const int cw = wv;
      const uint32_t ce = ev;
      if (c0 + 64 < cols) {  // the next chunk's loads run under this one's work
        wv = w[c0 + 64 + lane];
        ev = er[c0 + 64 + lane];
      }
      const uint32_t v = static_cast<uint32_t>(cw) + 2u * ce;
      uint64_t m = __ballot(cw < th);  // (rows past the index are INT_MAX)
      while (m) {
        const int src = __builtin_ctzll(m);
        if (cnt < static_cast<uint32_t>(cap) && lane == 0)
          cand_idx[qi * cap + cnt] = static_cast<uint32_t>(c0 + src);
        ++cnt;
        const uint32_t x = lane_value(v, src);
        m &= m - 1;
        if (x < ks.kth) {
          ks.insert(x, lane, k);
          th = q16_threshold(ks.kth, eq, rho);
          m &= __ballot(cw < th);
        }
      }
    }
  }
  if (lane < k) seed[qi * k + lane] = ks.b;
  if (lane == 0) cand_count[qi] = cnt;
}

// One level (knn_lists.hpp).  QW = 4: a workgroup takes a run of (query
// tile, row tile) pairs, as the FP64 form's scan does.  QW = 1 (one query
// tile): each of its wavefronts takes a run of row tiles of its own.
template <int QW>
__global__ __launch_bounds__(kSadThreads, 3) void l1q_scan_kernel(
    const uint32_t* __restrict__ codes, const uint32_t* __restrict__ er, int64_t n, int ldq, int ndw,
    const uint32_t* __restrict__ qcodes, const double* __restrict__ eqv, int64_t q,
    const uint32_t* __restrict__ seed, int k, double rho, Level lv, ScanOut<uint32_t> out) {
  __shared__ __align__(16) SadSmem<QW> sm;
  // per wavefront and query: threshold, entries so far and at the last look
  __shared__ int s_th[4][32];
  __shared__ uint32_t s_cnt[4][32], s_mark[4][32];
  const SadLane sl;
  const uint32_t grow = static_cast<uint32_t>(max(2 * k, 32));
  const int64_t rend = min(n, lv.row0 + lv.tiles * kListTile);
  const int64_t nqt = QW == 4 ? (q + 127) / 128 : 1;
  int64_t pos = static_cast<int64_t>(blockIdx.x) * lv.per * SadSmem<QW>::RW;
  const int64_t end = min(pos + lv.per * SadSmem<QW>::RW, nqt * lv.tiles);
  while (pos < end) {
    const int64_t qt = QW == 4 ? pos / lv.tiles : 0;
    const int64_t tb = pos - qt * lv.tiles;
    const int64_t te = QW == 4 ? min(lv.tiles, tb + (end - pos)) : tb + lv.per;
    const int list = QW == 4 ? static_cast<int>(blockIdx.x - qt * lv.tiles / lv.per)
                             : static_cast<int>(blockIdx.x) * 4 + sl.wave;
    const int64_t q0 = qt * 128 + (QW == 4 ? sl.wave * 32 : 0);  // the wavefront's first query
    const int64_t rb = lv.row0 + tb * kListTile;
    const int64_t mine = rb + (QW == 4 ? 0 : sl.wave * lv.per * kListTile);
    if (sl.lane < 32) {
      const int64_t qi = q0 + sl.lane;
      // queries past the batch or outside the domain take no part
      s_th[sl.wave][sl.lane] =
          qi < q && eqv[qi] < INFINITY ? q16_threshold(seed[qi * k + k - 1], eqv[qi], rho) : -0x7fffffff - 1;
      s_cnt[sl.wave][sl.lane] = 0u;
      s_mark[sl.wave][sl.lane] = 0u;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    auto slot_of = [&](int ql, uint32_t c) {
      return (q0 + ql) * out.entries + lv.entry0 + static_cast<int64_t>(list) * lv.cap + c;
    };
    sad_sweep<QW>(sm, codes, n, ldq, ndw, qcodes, q, QW == 4 ? qt * 128 : 0, rb,
                  lv.per * kListTile, te - tb, [&](int64_t t, SadAcc& acc) {
      const int64_t r0 = mine + t * kListTile;
      if (r0 >= rend) return;  // (a stream past the level's end)
      int e[8];
      tile_er(sl, er, r0, e);
      bool grown = false;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int ql = sl.query_of(i);
        const int th = s_th[sl.wave][ql];
        uint64_t some = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          acc[i][j] -= static_cast<uint32_t>(e[j]);  // W
          some |= __ballot(static_cast<int>(acc[i][j]) < th);
        }
        if (some == 0) continue;  // the whole wavefront
        uint64_t m[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          m[j] = __ballot(static_cast<int>(acc[i][j]) < th &&
                          r0 + sl.row_of(j >> 2, j & 3) < rend) & sl.peers();
        const uint32_t base = s_cnt[sl.wave][ql];
        uint32_t before = base;  // entries of the halves and lanes ahead
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          uint32_t c = before;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            c += __popcll(m[4 * h + r] & sl.below());
            before += __popcll(m[4 * h + r]);
          }
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if ((m[4 * h + r] >> sl.lane) & 1u) {
              if (c < static_cast<uint32_t>(lv.cap)) {
                const int64_t s = slot_of(ql, c);
                out.idx[s] = static_cast<uint32_t>(r0 + sl.row_of(h, r));
                out.u[s] = acc[i][4 * h + r] + 2u * static_cast<uint32_t>(e[4 * h + r]);  // V
              }
              ++c;
            }
        }
        if (sl.tr == 0) s_cnt[sl.wave][ql] = before;
        grown = grown || before - s_mark[sl.wave][ql] >= grow;
      }
      if (__ballot(grown) == 0) return;
      // lists that grew by `grow` since they were last looked at: their own
      // k-th V is a threshold too
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
      for (int ql = 0; ql < 32; ++ql) {
        const uint32_t c = s_cnt[sl.wave][ql];
        if (c - s_mark[sl.wave][ql] < grow) continue;  // the same in all lanes
        KSmallest<uint32_t> ks;
        ks.clear();
        ks.take(out.u + slot_of(ql, 0), min(c, static_cast<uint32_t>(lv.cap)), sl.lane, k);
        if (sl.lane == 0) {
          // past cap its list is lost (the sequential kernel takes the query):
          // no more rows for it
          const int th = c > static_cast<uint32_t>(lv.cap) ? -0x7fffffff - 1
                                                           : q16_threshold(ks.kth, eqv[q0 + ql], rho);
          if (th < s_th[sl.wave][ql]) s_th[sl.wave][ql] = th;
          s_mark[sl.wave][ql] = c;
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    });
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    if (sl.lane < 32 && q0 + sl.lane < q && list < lv.lists && mine < rend)
      out.count[(q0 + sl.lane) * out.lists + lv.list0 + list] = s_cnt[sl.wave][sl.lane];
    pos += te - tb;
    __syncthreads();  // the sweep's LDS is staged anew
    if (QW == 1) break;
  }
}

// Builds the 16-bit coded copy of an f32 index once (under its lock).  The
// form is taken when every value is finite with |v| <= 1e30 and the code step
// h (the smallest power of two with (max - min) / h <= 65534) is at most
// 1/64 of the mean |v|, so the bound's band (about d h) stays a few percent
// of a typical distance; otherwise, and for rows of more than 832 values, the
// index keeps the f32 scan.  The width limit is that of an earlier scan, which
// staged whole queries in LDS; a test holds that 900 values are declined.  This
// kernel would take up to 16,384 and be the faster form (f32 scan and codes: 300
// queries x 100,000 x 840: 28.9 and 1.2 ms; 1,000 x 20,000 x 4,096: 155 and 3.6; 50 x
// 5,000 x 9,000: 3.6 and 3.1; 5 x 2,000 x 32,000: 9.9 and 10.4).
constexpr int kQ16MaxLd = 832;

}  // namespace

int ensure_q16(sc_index* ix, bool* coded, hipStream_t s) {
  std::lock_guard<std::mutex> lk(*static_cast<std::mutex*>(ix->mu));
  *coded = ix->q16_state == 1;
  if (ix->q16_state != 0) return SC_OK;
  const int64_t n = static_cast<int64_t>(ix->n);
  const int d = static_cast<int>(ix->d), ld = static_cast<int>(ix->ld);
  if (n == 0 || d == 0 || ld > kQ16MaxLd) {
    ix->q16_state = 2;
    return SC_OK;
  }
  const float* rows = static_cast<const float*>(ix->rows);
  const int blocks = static_cast<int>(std::min<int64_t>(2048, (n + 15) / 16));
  DevBuf part;
  SC_HIP(part.alloc(sizeof(double) * 4 * blocks, s));
  hipLaunchKernelGGL(q16_range_kernel, dim3(blocks), dim3(256), 0, s, rows, n, d, ld,
                     part.as<double>());
  SC_HIP(hipGetLastError());
  std::vector<double> h(4 * static_cast<size_t>(blocks));
  SC_HIP(hipMemcpyAsync(h.data(), part.p, sizeof(double) * h.size(), hipMemcpyDeviceToHost, s));
  SC_HIP(hipStreamSynchronize(s));
  double mn = INFINITY, mx = -INFINITY, sum = 0.0, bad = 0.0;
  for (int b = 0; b < blocks; ++b) {
    mn = std::min(mn, h[4 * b]);
    mx = std::max(mx, h[4 * b + 1]);
    sum += h[4 * b + 2];
    bad = std::max(bad, h[4 * b + 3]);
  }
  if (bad != 0.0 || !(mn <= mx)) {
    ix->q16_state = 2;
    return SC_OK;
  }
  const double range = mx - mn;
  double step = std::ldexp(1.0, -100);
  if (range > 0.0) {
    int e = 0;
    (void)std::frexp(range / 65534.0, &e);  // range / 65534 < 2^e
    step = std::max(step, std::ldexp(1.0, e));
  }
  double lo = std::floor(mn / step) * step;
  while ((mx - lo) / step > 65535.0) {  // not reached for the step above
    step *= 2.0;
    lo = std::floor(mn / step) * step;
  }
  const double mean_abs = sum / (static_cast<double>(n) * d);
  if (range > 0.0 && step > mean_abs / 64.0) {
    ix->q16_state = 2;
    return SC_OK;
  }
  void* codes = nullptr;
  uint32_t* er = nullptr;
  SC_HIP(hipMalloc(&codes, sizeof(uint32_t) * static_cast<size_t>(n) * (ld / 2)));
  const int64_t npad = (n + kListTile - 1) / kListTile * kListTile;
  if (hipMalloc(reinterpret_cast<void**>(&er), sizeof(uint32_t) * npad) != hipSuccess) {
    (void)hipFree(codes);
    return hip_fail(hipErrorOutOfMemory, "hipMalloc(row code errors)");
  }
  hipLaunchKernelGGL(q16_rows_kernel, dim3(row_blocks(npad, 8, 256)), dim3(256), 0, s,
                     rows, n, npad, d, ld, lo, step, static_cast<uint32_t*>(codes), er);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) {
    (void)hipFree(codes);
    (void)hipFree(er);
    return hip_fail(e, "q16_rows_kernel");
  }
  ix->rows_q16 = codes;
  ix->err_q16 = er;
  ix->q16_lo = lo;
  ix->q16_step = step;
  ix->q16_state = 1;
  *coded = true;
  return SC_OK;
}

int knn_l1q_device(const sc_index* index, const float* d_queries, int64_t q, int k, int64_t* d_idx,
                   double* d_dist, uint32_t* d_count, hipStream_t s, sc_stats* stats) {
  const int64_t n = static_cast<int64_t>(index->n);
  const int ld = static_cast<int>(index->ld), d = static_cast<int>(index->d);
  const int ldq = ld / 2, ndw = (d + 1) / 2;
  const float* rows = static_cast<const float*>(index->rows);
  const uint32_t* codes = static_cast<const uint32_t*>(index->rows_q16);
  const uint32_t* er = index->err_q16;
  // rho >= (1 + eps) / (1 - eps), eps = 2^-24 + (d + 1) 2^-52
  const double rho = 1.0 + 3.0 * (5.9604644775390625e-08 + (d + 1.0) * 2.220446049250313e-16);
  const int64_t cols = std::min<int64_t>(kDenseRows, (n + kListTile - 1) / kListTile * kListTile);
  const std::vector<int64_t> edge = level_edges(n, cols);
  const int nlev = static_cast<int>(edge.size()) - 1;
  const int pre_cap = static_cast<int>(std::min<int64_t>(
      cols, static_cast<int64_t>(4.0 * expected_entrants(k, static_cast<double>(cols))) + 128));
  // Up to 32 queries would leave three quarters of a 128-query tile empty:
  // the wavefronts share the rows then (2,000,000 x 96 rows, 32 queries: 0.60 ms
  // against 0.86 with the wide tile, 1 query: 0.54 against 0.82).
  auto narrow = [](int64_t qn) { return qn <= 32; };
  // four workgroups per CU; narrow: two, of four pieces each
  auto plan = [&](int64_t qn, Level (&lv)[kMaxLevels], ScanOut<uint32_t>& o) {
    plan_levels(edge, qn, narrow(qn) ? 32 : 128, narrow(qn) ? 2048 : 1024, k, lv, o);
  };
  Lists<uint32_t> ls{};
  ls.nlevels = nlev;
  ls.pre_cap = pre_cap;
  const Batches batches = plan_batches<uint32_t>(
      q, plan,
      [&](const ScanOut<uint32_t>& o) {
        return 8.0 * o.entries + 4.0 * o.lists + 4.0 * pre_cap + 4.0 * (cols + k + ldq);
      },
      ls.lv, ls.out);
  const int64_t qb = batches.queries;
  DevBuf flags, olist, qcodes, qerr, dense, pidx, pcnt, cidx, cu, ccnt, seed;
  SC_HIP(flags.alloc(64, s));  // [0] listed queries, [2..3] candidate total (u64)
  SC_HIP(olist.alloc(sizeof(uint32_t) * qb, s));
  SC_HIP(qcodes.alloc(sizeof(uint32_t) * qb * ldq, s));
  SC_HIP(qerr.alloc(sizeof(double) * qb, s));
  SC_HIP(dense.alloc(sizeof(int) * qb * cols, s));
  SC_HIP(pidx.alloc(sizeof(uint32_t) * qb * pre_cap, s));
  SC_HIP(pcnt.alloc(sizeof(uint32_t) * qb, s));
  SC_HIP(seed.alloc(sizeof(uint32_t) * qb * k, s));
  SC_HIP(cidx.alloc(sizeof(uint32_t) * batches.entries, s));
  SC_HIP(cu.alloc(sizeof(uint32_t) * batches.entries, s));
  SC_HIP(ccnt.alloc(sizeof(uint32_t) * batches.lists, s));
  uint32_t* list_n = flags.as<uint32_t>();
  unsigned long long* total = reinterpret_cast<unsigned long long*>(flags.as<char>() + 8);
  hipLaunchKernelGGL(zero_words_kernel, dim3(1), dim3(64), 0, s, flags.as<uint32_t>(), int64_t{16});
  for (int64_t b0 = 0; b0 < q; b0 += qb) {
    const int64_t qn = std::min(qb, q - b0);
    const float* qs = d_queries + b0 * ld;
    if (qn != qb) plan(qn, ls.lv, ls.out);
    ls.pre_idx = pidx.as<uint32_t>();
    ls.pre_count = pcnt.as<uint32_t>();
    ls.out.idx = cidx.as<uint32_t>();
    ls.out.u = cu.as<uint32_t>();
    ls.out.count = ccnt.as<uint32_t>();
    hipLaunchKernelGGL(zero_words_kernel, dim3(1), dim3(64), 0, s, list_n, int64_t{1});
    hipLaunchKernelGGL(q16_queries_kernel, dim3(row_blocks(qn, 8, 256)), dim3(256), 0, s,
                       qs, qn, d, ld, index->q16_lo, index->q16_step, qcodes.as<uint32_t>(),
                       qerr.as<double>(), olist.as<uint32_t>(), list_n);
    SC_HIP(hipGetLastError());
    const unsigned sel = static_cast<unsigned>((qn + kSelectWaves - 1) / kSelectWaves);
    {
      ProfScope ps("knn_scan_q16", s);
      hipLaunchKernelGGL(l1q_dense_kernel,
                         dim3(static_cast<unsigned>((qn + 127) / 128), static_cast<unsigned>(cols / kListTile)),
                         dim3(kSadThreads), 0, s, codes, er, n, ldq, ndw, qcodes.as<uint32_t>(), qn,
                         cols, dense.as<int>());
      hipLaunchKernelGGL(l1q_select_dense_kernel, dim3(sel), dim3(64 * kSelectWaves), 0, s,
                         dense.as<int>(), cols, er, qerr.as<double>(), qn, k, rho, pre_cap,
                         pidx.as<uint32_t>(), pcnt.as<uint32_t>(), seed.as<uint32_t>());
      SC_HIP(hipGetLastError());
      if (nlev > 0) {
        const int64_t w = qn * ls.out.lists;
        hipLaunchKernelGGL(zero_words_kernel, dim3(static_cast<unsigned>(std::min<int64_t>(1024, (w + 255) / 256))),
                           dim3(256), 0, s, ls.out.count, w);
      }
      for (int i = 0; i < nlev; ++i) {
        const Level& lv = ls.lv[i];
        if (narrow(qn))
          hipLaunchKernelGGL(l1q_scan_kernel<1>, dim3(static_cast<unsigned>((lv.groups + 3) / 4)),
                             dim3(kSadThreads), 0, s, codes, er, n, ldq, ndw, qcodes.as<uint32_t>(),
                             qerr.as<double>(), qn, seed.as<uint32_t>(), k, rho, lv, ls.out);
        else
          hipLaunchKernelGGL(l1q_scan_kernel<4>, dim3(static_cast<unsigned>(lv.groups)),
                             dim3(kSadThreads), 0, s, codes, er, n, ldq, ndw, qcodes.as<uint32_t>(),
                             qerr.as<double>(), qn, seed.as<uint32_t>(), k, rho, lv, ls.out);
        if (i + 1 < nlev)
          hipLaunchKernelGGL(select_level_kernel<uint32_t>, dim3(sel), dim3(64 * kSelectWaves), 0, s, lv,
                             ls.out, qn, k, seed.as<uint32_t>());
        SC_HIP(hipGetLastError());
      }
    }
    {
      ProfScope ps("knn_mixed_rescore", s);
      launch_finish<float, kManhattan>(rows, ld, qs, qn, k, ls, d_idx + b0 * k, d_dist + b0 * k,
                                       d_count + b0, olist.as<uint32_t>(), list_n, stats ? total : nullptr, s);
      SC_HIP(hipGetLastError());
    }
    if (int rc = launch_serial_manhattan_f32(index, qs, k, olist.as<uint32_t>(), list_n, d_idx + b0 * k,
                                             d_dist + b0 * k, d_count + b0, s))
      return rc;
    if (stats) {
      uint64_t h[2] = {0, 0};
      SC_HIP(hipMemcpyAsync(h, flags.p, 16, hipMemcpyDeviceToHost, s));
      SC_HIP(hipStreamSynchronize(s));
      stats->overflow_queries += static_cast<uint32_t>(h[0]);
      if (b0 + qn >= q) {
        stats->candidates += h[1];
        stats->shortlist_rescored += h[1];
      }
    }
  }
  if (stats) stats->queries += static_cast<uint64_t>(q);
  return SC_OK;
}

}  // namespace sc
