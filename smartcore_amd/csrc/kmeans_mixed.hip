// Certified BF16-MFMA Lloyd step for f32 rows (sc_kmeans_run and
// sc_kmeans_batch_run, SC_MIXED): a label kernel, then a block-sums kernel.
//
// The label kernel runs four-wave workgroups over 128-row chunks, each wave
// 32 rows; a lane loads the values of its row that it feeds the MFMA
// straight from memory (no LDS stage), and the rows of the workgroup's next
// chunk are requested while the current one is labelled.  The centroid
// tables sit in LDS, loaded once per problem.
//
// Labels.  Each wave takes 32 rows of the chunk and splits them into three
// BF16 terms (x = xh + xm + xl + r, |r| <= 2^-24 |x|); the centroid tables
// hold the same split of v = RN_f32(-2c).  Six v_mfma_f32_32x32x16_bf16
// products per K step in three phases by weight, smallest first ((lo, hi),
// (hi, lo), (mid, mid) at 2^-16; (mid, hi), (hi, mid) at 2^-8; (hi, hi))
// plus ||c||^2 give, for every centroid, a_c ~ s_c - ||x||^2, where s_c is
// the f64 squared distance that KMeans::predict computes
// (kmeans.rs:338-346: x widened to f64, differences and squares in f64,
// summed in dimension order).  With
//   c1 = 5.3 * 2^-24 + (ld + 1 + 2.1 ld 2^-7 + 3.1 ld 2^-14) * 2.04 * 2^-24
// (representation errors of both operands, the f32 rounding of -2c and the
// dropped (mid, lo), (lo, mid), (lo, lo) products; FP32 accumulation at two
// ulps per add at each phase's scale) and
//   E = 2 c1 ||x|| max||c|| + 2^-20 (||x||^2 + max||c||^2)
// (the f32 norms, the final add and the f64 rounding of s_c), every c has
// |a_c - (s_c - ||x||^2)| <= E.  A row whose minimum a is the only value
// <= min a + 2E is certified: every other centroid has s_c strictly above
// the winner's, so the winner is the exact argmin.  Any other centroid with
// a_c <= min a + 2E is a candidate, and no non-candidate can be the argmin
// or tie with it.  An uncertified row is assigned among its candidates only:
// the wave computes each candidate's s_c with lanes = dimensions and a fixed
// tree (it differs from the sequential fold of the same terms by at most
// (ld + 6) ulps), and a best value below the runner-up by more than twice
// that is the exact argmin; near-exact ties take the reference's sequential
// fold and the lowest (value, index) -- the rule of the FP64 assign kernel
// (strict < in index order).  Rows that are not finite, or whose squared
// norm is at least 1e30 or below 1e-30 (but not zero), compute all k
// distances.  So the labels equal the FP64 form's on every input.
//
// Sums.  A second kernel reads each 2048-row block's labels, sorts the
// block's rows by label in LDS (stable: row order inside each cluster) and
// adds each cluster's run of rows in that order into f64 registers, lane =
// dimension.  That is the order of the FP64 form's partial kernel, so both
// forms write the same block partials bit for bit, and the shared reduce
// kernels give the same sums, centroids and distortions.
//
// Batched form.  Many independent problems (uneven n, d, k) run per Lloyd
// iteration as one persistent label launch per shape class over (problem,
// chunk) items (the classes one after another, most work first), one sums
// launch over every (problem, block), then the shared reduce kernels over
// every problem.  The problems go in two groups of about equal row bytes:
// the second group's rows are copied on a stream of their own while the
// first group iterates, and each group's iterations are captured in one
// hipGraph.  The label grid size is picked by timing the first iterations.
// Every problem gets bit-identical results to sc_kmeans_run on it alone.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "common.hpp"
#include "kmeans.hpp"
#include "metric.hpp"

namespace sc {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int NT = 256;  // threads of the helper kernels
constexpr uint32_t kUncert = 0xffffffffu;
constexpr double kKappa = 9.5367431640625e-07;   // 2^-20
constexpr size_t kLdsBudget = 150 * 1024;         // dynamic LDS one workgroup may take

// Shape class of the label kernel: k <= 32 KBM, padded dimension <= 16 KSM;
// W waves per workgroup, 32 rows each.
template <int KBM, int KSM, int W = 4>
struct Cfg {
  static constexpr int LD = 16 * KSM;                    // largest padded dimension
  static constexpr int KP = 32 * KBM;                    // largest padded k
  static constexpr int WAVES = W;                        // waves per workgroup
  static constexpr int NTH = 64 * WAVES;                 // threads per workgroup
  static constexpr int CR = 32 * WAVES;                  // rows per chunk
  static constexpr int DPL = (LD + 63) / 64;             // dimensions per lane
  static constexpr int LDA = LD + 8;                     // A-table row stride: 16 B of padding
  static constexpr size_t ATAB = sizeof(uint16_t) * KP * LDA;
  // LDS: c2 | A tables (hi | mid | lo)
  static constexpr size_t LABEL_LDS = sizeof(float) * KP + 3 * ATAB;
  // accumulator and row-value registers per lane
  static constexpr int LABEL_REGS = 16 * KBM + 8 * KSM;
  // waves per SIMD the label kernel is compiled for (EXACT: fixed loop
  // bounds, fewer live registers)
  static constexpr int label_waves(bool exact) {
    return LABEL_REGS < 32 ? 4 : (LABEL_REGS <= (exact ? 64 : 48) ? 3 : 2);
  }
  static_assert(kBlockRows % CR == 0, "a block is a whole number of chunks");
};

__device__ __forceinline__ uint32_t bf16_bits(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return u >> 16;
}

__device__ __forceinline__ bf16x8 as_frag(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

__device__ __forceinline__ bf16x8 load_frag(const uint16_t* p) {
  return as_frag(*reinterpret_cast<const u32x4*>(p));
}

__device__ __forceinline__ void lexmin_d(double& v, uint32_t& i, double v2, uint32_t i2) {
  if (v2 < v || (v2 == v && i2 < i)) {
    v = v2;
    i = i2;
  }
}

// s_c of KMeans::predict for one row (f32, stride 1) and one centroid (f64):
// the reference's sequential fold.
template <typename XP, typename CP>
__device__ __forceinline__ double exact_s(XP x, CP c, int ld) {
  double s = 0.0;
  for (int j = 0; j < ld; ++j) s = s + Term<double, kEuclid>::f(static_cast<double>(x[j]), c[j], 2.0);
  return s;
}

// Centroid index of bit `sl` (16 cb + v) of a lane in row half `half`.
__device__ __forceinline__ uint32_t slot_centroid(int sl, int half) {
  return static_cast<uint32_t>(32 * (sl >> 4) + 8 * ((sl & 15) >> 2) + 4 * half + (sl & 3));
}

// Rows of one label work item: one chunk of a four-wave workgroup.
constexpr int kSegRows = 128;

// The eight values of the lane's row that it feeds the MFMA in each K step.
template <int KSM, bool EXACT>
__device__ __forceinline__ void load_row_parts(const float* xr, int ks_n, int half,
                                               f32x4 (&xv)[KSM][2]) {
#pragma unroll
  for (int ks = 0; ks < KSM; ++ks)
    if (EXACT || ks < ks_n) {
      const auto s4 = to_global(reinterpret_cast<const f32x4*>(xr + 16 * ks + 8 * half));
      xv[ks][0] = s4[0];
      xv[ks][1] = s4[1];
    }
}

// Labels of rows [rb, re) of problem p (one chunk, 32 rows per wave), with
// the centroid tables of p in LDS and the lane's row values already in xv.
// next_xr (or null): the lane's row of the workgroup's next chunk, whose
// values are loaded into xv once this chunk's MFMAs have consumed them.
// EXACT: the problem has exactly KBM centroid blocks and KSM K steps.
template <int KBM, int KSM, bool EXACT, int W>
__device__ __forceinline__ void km_label_chunk(const KmProb& p, int64_t c0, int64_t re,
                                               f32x4 (&xv)[KSM][2], const float* next_xr,
                                               const unsigned char* smem,
                                               unsigned long long& fb) {
  using C = Cfg<KBM, KSM, W>;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int col = lane & 31;
  const int half = lane >> 5;
  const int k = p.k;
  const int ld = p.ld;
  const int kb = EXACT ? KBM : (k + 31) / 32;
  const int ks_n = EXACT ? KSM : ld / 16;
  const float* c2s = reinterpret_cast<const float*>(smem);
  const uint16_t* ahi = reinterpret_cast<const uint16_t*>(c2s + C::KP);
  const uint16_t* amd = ahi + C::KP * C::LDA;
  const uint16_t* alo = amd + C::KP * C::LDA;
  const float* rows = static_cast<const float*>(p.rows);
  const auto grows = to_global(rows);
  const auto cent = to_global(static_cast<const double*>(p.cent));
  auto frag = [&](const uint16_t* tab, int cb, int ks) -> bf16x8 {
    return load_frag(tab + (32 * cb + col) * C::LDA + 16 * ks + 8 * half);
  };
  const float cmax = to_global(p.cmax)[0];
  const float c2max = to_global(p.cmax)[1];
  // cross-term error constant, relative to sum |x_i| |v_i| <= ||x|| ||v||:
  // representation (both three-term residuals, the f32 rounding of -2c) and
  // the dropped mid x lo, lo x mid, lo x lo products (5.3 * 2^-24), and FP32
  // accumulation at two ulps per add: 3 ld adds at 2^-14 in the first phase,
  // 2 ld adds at 1.02 * 2^-7 in the second, ld + 1 adds at 1.02 in the last
  const double c1 = 5.3 * 5.9604644775390625e-08 +
                    (ld + 1.0 + 2.1 * ld * 0.0078125 + 3.1 * ld * 6.103515625e-05) * 2.04 *
                        5.9604644775390625e-08;
  // tree vs sequential f64 fold of the same ld non-negative terms
  const double dr = 2.0004 * (ld + 8.0) * 1.1102230246251565e-16;

  {
    const int64_t row = c0 + 32 * wave + col;
    const bool pvalid = row < re;
    // the lane's row (an in-range row for lanes past the end: their values
    // fed only their own MFMA columns, which are never used)
    const float* xr = rows + (pvalid ? row : c0) * ld;

    // ---- labels of this wave's 32 rows ----
    // Three MFMA phases by term weight, smallest first: (lo(c) hi(x),
    // hi(c) lo(x), mid(c) mid(x)) at 2^-16, (mid(c) hi(x), hi(c) mid(x)) at
    // 2^-8, then hi(c) hi(x).  Each phase splits the row's values again, so
    // no split is held across phases.
    float x2p = 0.0f;
    f32x16 acc[KBM];
#pragma unroll
    for (int cb = 0; cb < KBM; ++cb) acc[cb] = f32x16{};
    // the parts of dimensions 16 ks + 8 half .. + 7 of the lane's row, two
    // values per v_cvt_pk_bf16_f32 (round to nearest even); the differences
    // v - hi and (v - hi) - mid are exact in f32
    auto split_x = [&](int ks, int parts, bf16x8& xh, bf16x8& xm, bf16x8& xl, bool norms) {
      const f32x4 v0 = xv[ks][0];
      const f32x4 v1 = xv[ks][1];
      const float v[8] = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
      u32x4 H, M = {0u, 0u, 0u, 0u}, L = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x2 a = {v[2 * q], v[2 * q + 1]};
        const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector(a, bf16x2));
        H[q] = h;
        if (parts > 1) {
          const f32x2 e1 = {a[0] - __uint_as_float(h << 16), a[1] - __uint_as_float(h & 0xffff0000u)};
          const uint32_t m = __builtin_bit_cast(uint32_t, __builtin_convertvector(e1, bf16x2));
          M[q] = m;
          if (parts > 2) {
            const f32x2 e2 = {e1[0] - __uint_as_float(m << 16),
                              e1[1] - __uint_as_float(m & 0xffff0000u)};
            L[q] = __builtin_bit_cast(uint32_t, __builtin_convertvector(e2, bf16x2));
          }
        }
      }
      if (norms) {
#pragma unroll
        for (int t = 0; t < 8; ++t) x2p = fmaf(v[t], v[t], x2p);
      }
      xh = as_frag(H);
      xm = as_frag(M);
      xl = as_frag(L);
    };
#pragma unroll
    for (int ks = 0; ks < KSM; ++ks)
      if (EXACT || ks < ks_n) {
        bf16x8 xh, xm, xl;
        split_x(ks, 3, xh, xm, xl, true);
#pragma unroll
        for (int cb = 0; cb < KBM; ++cb)
          if (EXACT || cb < kb) {
            acc[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag(alo, cb, ks), xh, acc[cb], 0, 0, 0);
            acc[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag(ahi, cb, ks), xl, acc[cb], 0, 0, 0);
            acc[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag(amd, cb, ks), xm, acc[cb], 0, 0, 0);
          }
      }
    // a compiler-level memory barrier: the next phase loads its operands
    // again instead of keeping the previous phase's in registers
    asm volatile("" ::: "memory");
#pragma unroll
    for (int ks = 0; ks < KSM; ++ks)
      if (EXACT || ks < ks_n) {
        bf16x8 xh, xm, xl;
        split_x(ks, 2, xh, xm, xl, false);
#pragma unroll
        for (int cb = 0; cb < KBM; ++cb)
          if (EXACT || cb < kb) {
            acc[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag(amd, cb, ks), xh, acc[cb], 0, 0, 0);
            acc[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag(ahi, cb, ks), xm, acc[cb], 0, 0, 0);
          }
      }
    asm volatile("" ::: "memory");
#pragma unroll
    for (int ks = 0; ks < KSM; ++ks)
      if (EXACT || ks < ks_n) {
        bf16x8 xh, xm, xl;
        split_x(ks, 1, xh, xm, xl, false);
#pragma unroll
        for (int cb = 0; cb < KBM; ++cb)
          if (EXACT || cb < kb)
            acc[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag(ahi, cb, ks), xh, acc[cb], 0, 0, 0);
      }
    if (next_xr) load_row_parts<KSM, EXACT>(next_xr, ks_n, half, xv);
    const float x2 = x2p + __shfl_xor(x2p, 32);

    // a_c = ||c||^2 + acc; lane (col, half) holds centroids
    // 32 cb + 8 g + 4 half + r for v = 4 g + r, in increasing index order.
    // The row's minimum over both halves sets the threshold (NaN values are
    // passed over by the minimum and fail every comparison below)
    float amin = INFINITY;
#pragma unroll
    for (int cb = 0; cb < KBM; ++cb) {
      if (EXACT || cb < kb) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 c2q = *reinterpret_cast<const f32x4*>(c2s + 32 * cb + 8 * g + 4 * half);
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[cb][4 * g + r] += c2q[r];
          amin = fminf(amin, fminf(fminf(acc[cb][4 * g], acc[cb][4 * g + 1]),
                                   fminf(acc[cb][4 * g + 2], acc[cb][4 * g + 3])));
        }
      }
    }
    amin = fminf(amin, __shfl_xor(amin, 32));
    const double x2u = static_cast<double>(x2) * (1.0 + 6.103515625e-05) + 1e-300;
    const double E = 2.0 * c1 * sqrt(x2u) * static_cast<double>(cmax) * (1.0 + 9.5367431640625e-07) +
                     kKappa * (x2u + static_cast<double>(c2max));
    const float thr = __double2float_ru(static_cast<double>(amin) + 2.0 * E * (1.0 + 9.765625e-04));
    // The candidates a_c <= thr, counted per lane; the row is certified when
    // its two lanes hold exactly one between them.  That candidate is the
    // minimum, and its slot is the one the lane recorded.
    uint32_t ncl = 0;
    int aslot = -1;  // 16 cb + v of the lane's last candidate
#pragma unroll
    for (int cb = 0; cb < KBM; ++cb)
      if (EXACT || cb < kb) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          // le = a <= thr (false for NaN); aslot = le ? slot : aslot;
          // ncl += le -- one compare result, used while it is in VCC
          asm("v_cmp_le_f32 vcc, %2, %3\n\t"
              "v_cndmask_b32_e64 %1, %1, %4, vcc\n\t"
              "v_addc_co_u32 %0, vcc, 0, %0, vcc"
              : "+v"(ncl), "+v"(aslot)
              : "v"(acc[cb][v]), "v"(thr), "i"(16 * cb + v)
              : "vcc");
        }
      }
    const uint32_t ncand = ncl + static_cast<uint32_t>(__shfl_xor(static_cast<int>(ncl), 32));
    uint32_t aidx = aslot >= 0 ? slot_centroid(aslot, half) : kUncert;
    aidx = min(aidx, static_cast<uint32_t>(__shfl_xor(static_cast<int>(aidx), 32)));
    const bool single = ncand == 1;
    // a finite threshold keeps padding centroids (a = +inf) out of the
    // candidates; anything else takes the all-centroid path below.  A NaN
    // or infinite value makes ||x||^2 NaN or +inf, which fails x2 < 1e30;
    // rows with 0 < ||x||^2 < 1e-30 could lose split terms to underflow
    const bool sane = x2 < 1e30f && (x2 == 0.0f || x2 >= 1e-30f) && amin < INFINITY &&
                      thr < INFINITY;
    const bool certified = sane && single;
    const bool cand = pvalid && sane && !certified;
    uint64_t cm = 0;  // an uncertified row's candidates in this lane: bit 16 cb + v
    if (cand) {
#pragma unroll
      for (int cb = 0; cb < KBM; ++cb)
        if (EXACT || cb < kb) {
          uint32_t m16 = 0;
#pragma unroll
          for (int v = 0; v < 16; ++v) m16 |= static_cast<uint32_t>(acc[cb][v] <= thr) << v;
          cm |= static_cast<uint64_t>(m16) << (16 * cb);
        }
    }

    // Level 2: s of each candidate with lanes = dimensions and a fixed tree
    // over the lanes; the lane owning the candidate keeps its best and
    // second-best value.  The tree differs from the reference's sequential
    // fold of the same terms by at most (ld + 6) ulps of the sum, so a best
    // value below the runner-up by more than twice that is the exact argmin.
    double b1 = INFINITY, b2 = INFINITY;
    uint32_t bc = kUncert;
    {
      uint64_t work = cm;
      for (;;) {
        const uint64_t act = __ballot(work != 0);
        if (act == 0) break;
        const int L = __builtin_ctzll(act);
        const uint32_t wlo = __builtin_amdgcn_readlane(static_cast<uint32_t>(work), L);
        const uint32_t whi = __builtin_amdgcn_readlane(static_cast<uint32_t>(work >> 32), L);
        const int sl = __builtin_ctzll((static_cast<uint64_t>(whi) << 32) | wlo);
        if (lane == L) work &= work - 1;
        const uint32_t c = slot_centroid(sl, L >> 5);
        if (c >= static_cast<uint32_t>(k)) continue;  // never: padding has a = +inf
        const auto xs = grows + (c0 + 32 * wave + (L & 31)) * ld;
        const int64_t cofs = static_cast<int64_t>(c) * ld;
        double t = 0.0;
#pragma unroll
        for (int dd = 0; dd < C::DPL; ++dd) {
          const int j = lane + 64 * dd;
          if (j < ld) t = t + Term<double, kEuclid>::f(static_cast<double>(xs[j]), cent[cofs + j], 2.0);
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) t = t + __shfl_xor(t, off);
        if (lane == L) {
          if (t < b1 || (t == b1 && c < bc)) {
            b2 = b1;
            b1 = t;
            bc = c;
          } else if (t < b2) {
            b2 = t;
          }
        }
      }
    }
    bool ok2;
    {
      const double pb1 = __shfl_xor(b1, 32);
      const double pb2 = __shfl_xor(b2, 32);
      const uint32_t pc = __shfl_xor(bc, 32);
      double second;
      if (pb1 < b1 || (pb1 == b1 && pc < bc)) {
        second = fmin(b1, pb2);
        b1 = pb1;
        bc = pc;
      } else {
        second = fmin(pb1, b2);
      }
      ok2 = b1 < INFINITY && second * (1.0 - dr) > b1;
    }
    // Level 3 (near-exact ties): the reference fold for each candidate
    uint64_t cm3 = ok2 ? 0 : cm;
    double bs = INFINITY;
    uint32_t bi = kUncert;
    while (__ballot(cm3 != 0)) {
      if (cm3 != 0) {
        const int sl = __builtin_ctzll(cm3);
        cm3 &= cm3 - 1;
        const uint32_t c = slot_centroid(sl, half);
        if (c < static_cast<uint32_t>(k))
          lexmin_d(bs, bi, exact_s(to_global(xr), cent + static_cast<int64_t>(c) * ld, ld), c);
      }
    }
    {
      const double v2 = __shfl_xor(bs, 32);
      const uint32_t i2 = __shfl_xor(bi, 32);
      lexmin_d(bs, bi, v2, i2);
    }
    if (half == 0 && pvalid && sane) {
      uint32_t lb = aidx;
      if (cand) lb = ok2 ? bc : (bs < DBL_MAX ? bi : 0u);
      to_global(p.labels)[row] = lb;
    }
    // rows outside the bound's domain: all k centroids, lanes = centroids
    uint64_t um = __ballot(half == 0 && pvalid && !sane);
    fb += static_cast<unsigned long long>(__popcll(__ballot(half == 0 && pvalid && !certified)));
    while (um) {
      const int q = __builtin_ctzll(um);
      um &= um - 1;
      const auto x = grows + (c0 + 32 * wave + q) * ld;
      double bv = INFINITY;
      uint32_t bj = kUncert;
      for (int c = lane; c < k; c += 64)
        lexmin_d(bv, bj, exact_s(x, cent + static_cast<int64_t>(c) * ld, ld), static_cast<uint32_t>(c));
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) {
        const double v2 = __shfl_xor(bv, off);
        const uint32_t i2 = __shfl_xor(bj, off);
        lexmin_d(bv, bj, v2, i2);
      }
      // kmeans.rs:334-347: min starts at f64::MAX; nothing below it keeps 0
      if (lane == 0) to_global(p.labels)[c0 + 32 * wave + q] = bv < DBL_MAX ? bj : 0u;
    }
  }
}

// Persistent label kernel over (problem, chunk) items of one shape class;
// with items == nullptr the launch covers every chunk of problem 0.  The
// centroid tables are loaded into LDS when the problem changes; the rows of
// the workgroup's next item are requested while the current one is
// labelled when both belong to the same problem.
template <int KBM, int KSM, bool EXACT, int W>
__global__ __launch_bounds__((Cfg<KBM, KSM, W>::NTH), (Cfg<KBM, KSM, W>::label_waves(EXACT))) void km_label_kernel(
    const KmProb* __restrict__ P, const uint2* __restrict__ items, int64_t nitems) {
  using C = Cfg<KBM, KSM, W>;
  static_assert(C::CR == kSegRows, "one chunk per item");
  extern __shared__ __align__(16) unsigned char smem[];
  float* c2s = reinterpret_cast<float*>(smem);
  uint16_t* ahi = reinterpret_cast<uint16_t*>(c2s + C::KP);
  uint16_t* amd = ahi + C::KP * C::LDA;
  uint16_t* alo = amd + C::KP * C::LDA;
  const int tid = threadIdx.x;
  const int col = tid & 31;
  const int half = (tid & 63) >> 5;
  const int wave = tid >> 6;
  unsigned long long fb = 0;
  int cur = -1;
  bool skip = false;
  bool have = false;  // xv holds the rows of item `it`
  KmState* st = nullptr;
  f32x4 xv[KSM][2];
  auto item = [&](int64_t it, int& i, int64_t& c0) {
    i = items ? static_cast<int>(items[it].x) : 0;
    c0 = (items ? static_cast<int64_t>(items[it].y) : it) * kSegRows;
  };
  auto lane_row = [&](const KmProb& q, int64_t c0) -> const float* {
    const int64_t row = min(c0 + 32 * wave + col, q.n - 1);
    return static_cast<const float*>(q.rows) + row * q.ld;
  };
  for (int64_t it = blockIdx.x; it < nitems; it += gridDim.x) {
    int i;
    int64_t c0;
    item(it, i, c0);
    const KmProb p = P[i];
    if (i != cur) {
      if (st && fb && (tid & 63) == 0) atomicAdd(&st->fallback, fb);
      fb = 0;
      // every workgroup of this launch sees the same value: the flag only
      // changes in the final reduce kernel
      skip = *reinterpret_cast<volatile uint32_t*>(&p.st->done) != 0;
      if (!skip) {
        __syncthreads();  // nobody reads the previous problem's tables
        for (int e = tid; e < C::KP; e += C::NTH) c2s[e] = e < p.kpad ? to_global(p.c2f)[e] : INFINITY;
        for (int e = tid; e < C::KP * C::LD / 8; e += C::NTH) {
          const int r = e / (C::LD / 8), j8 = e % (C::LD / 8);
          const bool in = r < p.kpad && 8 * j8 < p.ld;
          const int64_t src = static_cast<int64_t>(r) * p.ld + 8 * j8;
          const u32x4 z = {0u, 0u, 0u, 0u};
          const int dst = r * C::LDA + 8 * j8;
          *reinterpret_cast<u32x4*>(ahi + dst) =
              in ? *to_global(reinterpret_cast<const u32x4*>(p.bhi + src)) : z;
          *reinterpret_cast<u32x4*>(amd + dst) =
              in ? *to_global(reinterpret_cast<const u32x4*>(p.bmd + src)) : z;
          *reinterpret_cast<u32x4*>(alo + dst) =
              in ? *to_global(reinterpret_cast<const u32x4*>(p.blo + src)) : z;
        }
        __syncthreads();
      }
      cur = i;
      st = p.st;
    }
    if (skip) continue;
    const int ks_n = EXACT ? KSM : p.ld / 16;
    if (!have) load_row_parts<KSM, EXACT>(lane_row(p, c0), ks_n, half, xv);
    // the next item's rows, when it is of the same problem
    const float* next_xr = nullptr;
    const int64_t nit = it + gridDim.x;
    if (nit < nitems) {
      int ni;
      int64_t nc0;
      item(nit, ni, nc0);
      if (ni == i) next_xr = lane_row(p, nc0);
    }
    have = next_xr != nullptr;
    km_label_chunk<KBM, KSM, EXACT, W>(p, c0, min<int64_t>(c0 + kSegRows, p.n), xv, next_xr, smem,
                                       fb);
  }
  // each wave adds its own count
  if (st && fb && (tid & 63) == 0) atomicAdd(&st->fallback, fb);
}

// ---- block partial sums from the labels ----
// One workgroup per (problem, block) item.  The block's rows are sorted by
// label (stable: row order inside each cluster) in LDS; then wave w adds the
// runs of clusters w, w + kSumWaves, ... one at a time into one f64
// accumulator per dimension, loading kSumBatch rows of a run at once.  The
// adds of each cluster are its rows in row order from +0.0 -- the order the
// FP64 form's partial kernel uses -- so both forms write the same block
// partials bit for bit.
constexpr int kSumWaves = 8;
constexpr int kSumThreads = 64 * kSumWaves;
// rows of a run in flight (registers: half as many of f64)
template <typename T>
constexpr int kSumBatch = sizeof(T) == 4 ? 32 : 16;
constexpr int kSumMaxK = 128;
constexpr int kSumGroups = kBlockRows / 64 / kSumWaves;  // 64-row groups per wave

// The runs of rows of up to 64 / G values: a load takes G rows at once (lane
// group g of 64 / G lanes holds row G t + g), so NB loads keep G NB rows in
// flight, and they go through the wavefront's LDS tile to be added in row
// order, one LDS read per row and dimension.  Rows past the run's end are
// stored as +0.0, which changes no bit of a sum that starts at +0.0 (it is
// never -0.0), so the adds need no test.  One row per load leaves most lanes
// idle and a run's chain bound by latency: 100,000 x 16 f64 rows in 10
// clusters took 40 us a step that way and take 17 (22 with the rows brought
// across the lanes by shuffles).
constexpr int kPackLoads = 16;
template <typename T, int G, typename Rows, typename Sums, typename Counts>
__device__ __forceinline__ void sum_runs_packed(Rows rows, int ld, int d, int k, int wave, int lane,
                                                const uint16_t* perm, const uint32_t* start, T* tile,
                                                Sums psum, Counts pcount) {
  constexpr int LW = 64 / G;
  constexpr int NR = G * kPackLoads;  // rows of a batch
  const int g = lane / LW, jl = lane % LW;
  const int j = min(jl, ld - 1);  // (past ld: a value that is never stored)
  for (int c = wave; c < k; c += kSumWaves) {
    const int e0 = static_cast<int>(start[c]), e1 = static_cast<int>(start[c + 1]);
    double acc = 0.0;
    for (int e = e0; e < e1; e += NR) {
      const int nv = e1 - e;
      T x[kPackLoads];
#pragma unroll
      for (int t = 0; t < kPackLoads; ++t)
        x[t] = rows[static_cast<int64_t>(perm[min(e + t * G + g, e1 - 1)]) * ld + j];
#pragma unroll
      for (int t = 0; t < kPackLoads; ++t)
        tile[(t * G + g) * LW + jl] = t * G + g < nv ? x[t] : T(0);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int t0 = 0; t0 < NR; t0 += 16) {
        if (t0 < nv) {
          T v[16];
#pragma unroll
          for (int t = 0; t < 16; ++t) v[t] = tile[(t0 + t) * LW + jl];
#pragma unroll
          for (int t = 0; t < 16; ++t) acc = acc + static_cast<double>(v[t]);
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    if (lane < d) psum[static_cast<int64_t>(c) * d + lane] = acc;
    if (lane == 0) pcount[c] = static_cast<uint32_t>(e1 - e0);
  }
}

// T: the rows' type.  DPL: dimensions per lane (2 when some row is wider than
// 64 values).  PACK: narrow rows in few clusters take the packed runs (whose
// tiles cost LDS): a block's runs average at least 64 rows there.
constexpr int kPackMaxK = 32;
constexpr int kPackTile = 64 * kPackLoads;  // values: NR rows of LW
template <typename T, int DPL, bool PACK>
__global__ __launch_bounds__(kSumThreads, DPL == 1 && !(PACK && sizeof(T) == 8) ? 4 : 2) void km_sums_kernel(
    const KmProb* __restrict__ P, const uint2* __restrict__ items, int64_t nitems) {
  __shared__ T tiles[PACK ? kSumWaves * kPackTile : 1];
  __shared__ uint32_t lab[kBlockRows];
  __shared__ uint16_t perm[kBlockRows];
  __shared__ uint32_t pos[kSumWaves][kSumMaxK];
  __shared__ uint32_t start[kSumMaxK + 1];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  for (int64_t it = blockIdx.x; it < nitems; it += gridDim.x) {
    const int i = items ? static_cast<int>(items[it].x) : 0;
    const int64_t b = items ? static_cast<int64_t>(items[it].y) : it;
    const KmProb p = P[i];
    if (*reinterpret_cast<volatile uint32_t*>(&p.st->done)) continue;
    const int k = p.k, d = p.d, ld = p.ld;
    const int64_t r0 = b * kBlockRows;
    const int nr = static_cast<int>(min<int64_t>(kBlockRows, p.n - r0));
    const auto labels = to_global(static_cast<const uint32_t*>(p.labels)) + r0;
    for (int e = tid; e < kBlockRows; e += kSumThreads) lab[e] = e < nr ? labels[e] : kUncert;
    for (int e = tid; e < kSumWaves * kSumMaxK; e += kSumThreads) (&pos[0][0])[e] = 0u;
    __syncthreads();
    // per 64-row group: the lanes holding the same label (eight bits: labels
    // are below 128, rows past the end get 255), the lane's rank among them
    // and their number; wave w's groups are rows 64 (4w) .. 64 (4w + 4)
    uint32_t key[kSumGroups], rk[kSumGroups], ng[kSumGroups];
#pragma unroll
    for (int gi = 0; gi < kSumGroups; ++gi) {
      const int g = kSumGroups * wave + gi;
      const uint32_t l = lab[64 * g + lane];
      const uint32_t kk = l < static_cast<uint32_t>(k) ? l : 0xffu;
      uint64_t eq = ~0ull;
#pragma unroll
      for (int bit = 0; bit < 8; ++bit) {
        const bool on = (kk >> bit) & 1u;
        const uint64_t B = __ballot(on);
        eq &= on ? B : ~B;
      }
      key[gi] = kk;
      rk[gi] = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(eq >> 32),
                                         __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(eq), 0u));
      ng[gi] = static_cast<uint32_t>(__popcll(eq));
      if (kk < static_cast<uint32_t>(k) && rk[gi] == 0) pos[wave][kk] += ng[gi];
    }
    __syncthreads();
    // cluster starts, and the first position of each wave's rows of each
    // cluster (wave 0; lane = clusters 2 lane, 2 lane + 1)
    if (wave == 0) {
      const int ca = 2 * lane, cb = 2 * lane + 1;
      uint32_t ha[kSumWaves], hb[kSumWaves], ta = 0, tb = 0;
#pragma unroll
      for (int w = 0; w < kSumWaves; ++w) {
        ha[w] = ca < k ? pos[w][ca] : 0u;
        hb[w] = cb < k ? pos[w][cb] : 0u;
        ta += ha[w];
        tb += hb[w];
      }
      uint32_t incl = ta + tb;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const uint32_t v = __shfl_up(incl, off);
        if (lane >= off) incl += v;
      }
      uint32_t sa = incl - ta - tb, sb = sa + ta;
      if (ca < k) start[ca] = sa;
      if (cb < k) start[cb] = sb;
      if (lane == 63) start[k] = incl;
#pragma unroll
      for (int w = 0; w < kSumWaves; ++w) {
        if (ca < k) pos[w][ca] = sa;
        if (cb < k) pos[w][cb] = sb;
        sa += ha[w];
        sb += hb[w];
      }
    }
    __syncthreads();
    // stable scatter, the wave's groups in row order
#pragma unroll
    for (int gi = 0; gi < kSumGroups; ++gi) {
      const int g = kSumGroups * wave + gi;
      if (key[gi] < static_cast<uint32_t>(k)) {
        perm[pos[wave][key[gi]] + rk[gi]] = static_cast<uint16_t>(64 * g + lane);
        if (rk[gi] == 0) pos[wave][key[gi]] += ng[gi];
      }
    }
    __syncthreads();
    // the runs
    const int64_t kd = static_cast<int64_t>(k) * d;
    const auto psum = to_global(p.psum) + b * kd;
    const auto rows = to_global(static_cast<const T*>(p.rows)) + r0 * ld;
    if constexpr (PACK) {
      T* tile = tiles + wave * kPackTile;
      if (ld <= 16)
        sum_runs_packed<T, 4>(rows, ld, d, k, wave, lane, perm, start, tile, psum, to_global(p.pcount) + b * k);
      else
        sum_runs_packed<T, 2>(rows, ld, d, k, wave, lane, perm, start, tile, psum, to_global(p.pcount) + b * k);
    } else {
    // two runs at a time: clusters c and c + kSumWaves, kSumBatch rows of
    // each requested before either is added
    const int j0 = min(lane, ld - 1), j1 = min(lane + 64, ld - 1);
    for (int c = wave; c < k; c += 2 * kSumWaves) {
      const int cc[2] = {c, c + kSumWaves};
      int e[2], e1[2];
      double acc[2][2] = {{0.0, 0.0}, {0.0, 0.0}};
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        e[u] = cc[u] < k ? static_cast<int>(start[cc[u]]) : 0;
        e1[u] = cc[u] < k ? static_cast<int>(start[cc[u] + 1]) : 0;
      }
      while (e[0] < e1[0] || e[1] < e1[1]) {
        int nv[2];
        T x[2][kSumBatch<T>][DPL];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          nv[u] = max(0, min(kSumBatch<T>, e1[u] - e[u]));
          const uint32_t mine = lane < nv[u] ? perm[e[u] + lane] : 0u;
          // lanes at or past ld read an in-row value that is never stored
#pragma unroll
          for (int t = 0; t < kSumBatch<T>; ++t) {
            const uint32_t r = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(mine), t));
            x[u][t][0] = rows[static_cast<int64_t>(r) * ld + j0];
            if (DPL > 1) x[u][t][1] = rows[static_cast<int64_t>(r) * ld + j1];
          }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
          for (int t = 0; t < kSumBatch<T>; ++t)
            if (t < nv[u]) {  // (the same in the whole wavefront: a scalar branch)
              acc[u][0] = acc[u][0] + static_cast<double>(x[u][t][0]);
              if (DPL > 1) acc[u][1] = acc[u][1] + static_cast<double>(x[u][t][1]);
            }
          e[u] += nv[u];
        }
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
        if (cc[u] < k) {
          if (lane < d) psum[static_cast<int64_t>(cc[u]) * d + lane] = acc[u][0];
          if (DPL > 1 && lane + 64 < d) psum[static_cast<int64_t>(cc[u]) * d + lane + 64] = acc[u][1];
          if (lane == 0)
            to_global(p.pcount)[b * k + cc[u]] = start[cc[u] + 1] - start[cc[u]];
        }
    }
    }
    __syncthreads();  // LDS is rewritten by the next item
  }
}

// Shape classes: KBM in {1, 2, 4}, KSM in {1, 2, 4, 8}.
int kbm_of(int k) { return k <= 32 ? 1 : (k <= 64 ? 2 : 4); }
int ksm_of(int ld) { return ld <= 16 ? 1 : (ld <= 32 ? 2 : (ld <= 64 ? 4 : 8)); }

// Whether a shape class's centroid tables fit one workgroup's LDS.
bool class_fits(int k, int ld) {
  if (k < 1 || k > kSumMaxK || ld > 128) return false;
  const int kbm = kbm_of(k), ksm = ksm_of(ld);
#define SC_KM_FIT(A, B) \
  if (kbm == A && ksm == B) return Cfg<A, B, 4>::LABEL_LDS <= kLdsBudget;
  SC_KM_FIT(1, 1) SC_KM_FIT(1, 2) SC_KM_FIT(1, 4) SC_KM_FIT(1, 8)
  SC_KM_FIT(2, 1) SC_KM_FIT(2, 2) SC_KM_FIT(2, 4) SC_KM_FIT(2, 8)
  SC_KM_FIT(4, 1) SC_KM_FIT(4, 2) SC_KM_FIT(4, 4) SC_KM_FIT(4, 8)
#undef SC_KM_FIT
  return false;
}

template <int KBM, int KSM, int W>
int launch_label_class(const KmProb* dP, const uint2* items, int64_t nitems, unsigned grid,
                       bool exact, hipStream_t s) {
  using C = Cfg<KBM, KSM, W>;
  const size_t lds = C::LABEL_LDS;
  const dim3 block(C::NTH);
  // allow the largest dynamic LDS this class can ask for (once per kernel)
  static const bool attr = [] {
    const int mx = static_cast<int>(kLdsBudget);
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&km_label_kernel<KBM, KSM, true, W>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, mx);
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&km_label_kernel<KBM, KSM, false, W>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, mx);
    return true;
  }();
  (void)attr;
  if (exact)
    hipLaunchKernelGGL((km_label_kernel<KBM, KSM, true, W>), dim3(grid), block, lds, s, dP, items,
                       nitems);
  else
    hipLaunchKernelGGL((km_label_kernel<KBM, KSM, false, W>), dim3(grid), block, lds, s, dP, items,
                       nitems);
  SC_HIP(hipGetLastError());
  return SC_OK;
}

// Workgroups of a class's label kernel one CU holds.
template <int KBM, int KSM, int W>
int label_groups_per_cu(bool exact) {
  using C = Cfg<KBM, KSM, W>;
  const int by_waves = C::label_waves(exact) * 4 / W;
  const int by_lds = static_cast<int>(160 * 1024 / C::LABEL_LDS);
  return std::max(1, std::min(by_waves, by_lds));
}

// mult: workgroups per CU in the grid (0: as many as one CU holds).  The
// grid is trimmed so that every workgroup gets the same number of items.
int launch_label(int kbm, int ksm, int mult, const KmProb* dP, const uint2* items,
                 int64_t nitems, bool exact, int cus, hipStream_t s) {
  auto grid_of = [&](int per) {
    const int64_t g = std::max<int64_t>(1, std::min<int64_t>(nitems, static_cast<int64_t>(mult ? mult : per) * cus));
    const int64_t each = (nitems + g - 1) / g;
    return static_cast<unsigned>(std::max<int64_t>(1, (nitems + each - 1) / each));
  };
#define SC_KM_CASE(A, B)                                                                  \
  if (kbm == A && ksm == B)                                                               \
    return launch_label_class<A, B, 4>(dP, items, nitems,                                \
                                       grid_of(label_groups_per_cu<A, B, 4>(exact)), exact, s);
  SC_KM_CASE(1, 1) SC_KM_CASE(1, 2) SC_KM_CASE(1, 4) SC_KM_CASE(1, 8)
  SC_KM_CASE(2, 1) SC_KM_CASE(2, 2) SC_KM_CASE(2, 4) SC_KM_CASE(2, 8)
  SC_KM_CASE(4, 1) SC_KM_CASE(4, 2) SC_KM_CASE(4, 4) SC_KM_CASE(4, 8)
#undef SC_KM_CASE
  return fail(SC_ERR_UNSUPPORTED, "k-means MFMA form: unsupported shape");
}

// ldmax: the widest padded row among the items' problems.
template <typename T>
int launch_sums(const KmProb* dP, const uint2* items, int64_t nitems, int ldmax, int k, int cus,
                hipStream_t s) {
  const unsigned grid = static_cast<unsigned>(std::max<int64_t>(1, std::min<int64_t>(nitems, 4 * cus)));
  // the packed form for a single problem only: a batch's launch holds every
  // shape, and the tiles' LDS would cost its many-cluster problems occupancy
  if (ldmax > 64)
    hipLaunchKernelGGL((km_sums_kernel<T, 2, false>), dim3(grid), dim3(kSumThreads), 0, s, dP, items, nitems);
  else if (!items && ldmax <= 32 && k <= kPackMaxK)
    hipLaunchKernelGGL((km_sums_kernel<T, 1, true>), dim3(grid), dim3(kSumThreads), 0, s, dP, items, nitems);
  else
    hipLaunchKernelGGL((km_sums_kernel<T, 1, false>), dim3(grid), dim3(kSumThreads), 0, s, dP, items, nitems);
  SC_HIP(hipGetLastError());
  return SC_OK;
}

int device_cus() {
  static int cached[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cached[dev] == 0) {
    hipDeviceProp_t prop;
    cached[dev] = hipGetDeviceProperties(&prop, dev) == hipSuccess && prop.multiProcessorCount > 0
                      ? prop.multiProcessorCount
                      : 256;
  }
  return cached[dev];
}

}  // namespace

bool kmeans_mixed_supported(const sc_index* ix, int k) {
  return ix->dtype == SC_F32 && class_fits(k, static_cast<int>(ix->ld));
}

bool kmeans_sorted_sums_supported(int k, int ld) { return k <= kSumMaxK && ld <= 128; }

int kmeans_sorted_sums_launch(const sc_index* ix, KmWork& w, hipStream_t s) {
  const int ld = w.p.ld, cus = device_cus();
  return ix->dtype == SC_F64 ? launch_sums<double>(w.dprob, nullptr, w.p.nb, ld, w.p.k, cus, s)
                             : launch_sums<float>(w.dprob, nullptr, w.p.nb, ld, w.p.k, cus, s);
}

int kmeans_mixed_step_launch(const sc_index* ix, KmWork& w, hipStream_t s) {
  if (w.p.nb == 0) return SC_OK;
  const int k = w.p.k, ld = w.p.ld;
  const int kbm = kbm_of(k), ksm = ksm_of(ld);
  const bool exact = (k + 31) / 32 == kbm && ld / 16 == ksm;
  const int cus = device_cus();
  const int64_t nseg = (w.p.n + kSegRows - 1) / kSegRows;
  ProfScope ps("kmeans_mixed_assign", s);
  if (int rc = launch_label(kbm, ksm, 0, w.dprob, nullptr, nseg, exact, cus, s)) return rc;
  return launch_sums<float>(w.dprob, nullptr, w.p.nb, ld, w.p.k, cus, s);
}

// ------------------------------------------------------------------ batch
namespace {

__global__ void kmb_init_kernel(const KmProb* __restrict__ P, int count) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  KmState* st = P[i].st;
  st->distortion = DBL_MAX;
  st->dist = 0.0;
  st->x2total = 0.0;
  st->iters = 0;
  st->done = 0;
  st->fallback = 0;
  *P[i].arrive = 0u;
}

// The shift mu of every problem: its first row, non-finite values as 0 (as
// the single-problem mu kernel).
__global__ void kmb_mu_kernel(const KmProb* __restrict__ P, int count) {
  const KmProb p = P[blockIdx.x];
  const float* rows = static_cast<const float*>(p.rows);
  for (int j = threadIdx.x; j < p.ld; j += blockDim.x) {
    const double v = p.n > 0 ? static_cast<double>(rows[j]) : 0.0;
    p.mu[j] = isfinite(v) ? v : 0.0;
  }
}

// ||x - mu||^2 per (problem, block): same order as the single-problem x2
// kernel.
__global__ __launch_bounds__(NT) void kmb_x2_kernel(const KmProb* __restrict__ P,
                                                    const uint2* __restrict__ items, int64_t nitems) {
  __shared__ double red[NT];
  const int tid = threadIdx.x;
  for (int64_t it = blockIdx.x; it < nitems; it += gridDim.x) {
    const KmProb p = P[items[it].x];
    const int64_t b = items[it].y;
    const float* rows = static_cast<const float*>(p.rows);
    const int64_t r0 = b * kBlockRows;
    double s = 0.0;
    for (int j = 0; j < kBlockRows / NT; ++j) {
      const int64_t r = r0 + tid * (kBlockRows / NT) + j;
      if (r < p.n) s = s + row_shift_x2(rows + r * p.ld, p.mu, p.ld);
    }
    red[tid] = s;
    __syncthreads();
    for (int w = NT / 2; w >= 1; w >>= 1) {
      if (tid < w) red[tid] = red[tid] + red[tid + w];
      __syncthreads();
    }
    if (tid == 0) p.x2block[b] = red[0];
    __syncthreads();
  }
}

__global__ void kmb_x2_total_kernel(const KmProb* __restrict__ P, int count) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const KmProb p = P[i];
  double s = 0.0;
  for (int64_t b = 0; b < p.nb; ++b) s = s + p.x2block[b];
  p.st->x2total = s;
}

struct Klass {
  int kbm, ksm;
  bool exact;
  int kmax = 0, ldmax = 0;
  std::vector<uint2> items;
  size_t at = 0;  // offset of the items in the call's item buffer
};

// Consecutive problems of one batched call whose rows go up together; the
// group's iterations run while the next group's rows are copied.  Its items
// hold problem indices relative to the group's first problem.
struct Group {
  size_t first = 0, count = 0;
  std::vector<uint2> all;  // (problem, 2048-row block), block-major
  size_t all_at = 0;       // offset of `all` in the call's item buffer
  std::map<int, Klass> klass;
  KmItems red;
  int ldmax = 0;
  int64_t rows = 0;
  int waves = 0, mult = 0;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  Group() = default;
  Group(const Group&) = delete;
  Group& operator=(const Group&) = delete;
  ~Group() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
  }
};

// Problem groups per batched call, and the fewest row bytes a group holds.
// Each group adds about 0.35 ms of fixed work per iteration (its own label,
// sums and reduce launches): on 512 problems (2.7 GB of rows, 20 iterations)
// calls took 111 / 95 / 98 / 100 ms with 1 / 2 / 3 / 4 groups.
constexpr int64_t kUploadGroups = 2;
constexpr int64_t kUploadGroupBytes = int64_t{64} << 20;

// The batched form's launch shape for a set of problems: label workgroups
// per CU (four waves each), and the waves per workgroup it was timed with.
struct TuneEntry {
  std::vector<int64_t> key;
  int waves, mult;
};
std::mutex g_tune_mu;
std::vector<TuneEntry> g_tune;

}  // namespace

}  // namespace sc

using namespace sc;

extern "C" int sc_kmeans_batch_run(const sc_kmeans_problem* problems, size_t count, sc_dtype dtype,
                                   size_t max_iter, sc_mode mode, double* centroids_out,
                                   uint32_t* labels_out, uint64_t* sizes_out,
                                   double* distortion_out, uint32_t* iters_out) {
  clear_error();
  if (count == 0) return SC_OK;
  if (!problems || !centroids_out || !labels_out || !sizes_out || !distortion_out || !iters_out)
    return fail(SC_PARAMETERS_ERROR, "null argument");
  if (max_iter == 0)
    return fail(SC_FIT_FAILED, "invalid maximum number of iterations: " + std::to_string(max_iter));
  if (dtype != SC_F64 && dtype != SC_F32) return fail(SC_ERR_UNSUPPORTED, "dtype must be f64 or f32");
  for (size_t i = 0; i < count; ++i) {
    if (problems[i].k < 2)
      return fail(SC_FIT_FAILED, "invalid number of clusters: " + std::to_string(problems[i].k));
    if (problems[i].n == 0 || !problems[i].rows || !problems[i].init_centroids)
      return fail(SC_PARAMETERS_ERROR, "problem " + std::to_string(i) + " has no rows");
  }
  int dev = 0;
  SC_HIP(hipGetDevice(&dev));
  hipStream_t s = stream_for_device(dev);

  bool batched = mode == SC_MIXED && dtype == SC_F32;
  for (size_t i = 0; i < count && batched; ++i)
    if (!class_fits(static_cast<int>(std::min<size_t>(problems[i].k, 1u << 20)),
                    static_cast<int>(std::min<size_t>(padded_dim(problems[i].d), 1u << 20))))
      batched = false;

  if (!batched) {
    // the FP64 form, one problem at a time (the comparator of the batch)
    size_t co = 0, lo = 0, so = 0;
    for (size_t i = 0; i < count; ++i) {
      const sc_kmeans_problem& pr = problems[i];
      sc_index* ix = nullptr;
      if (int rc = sc_index_create(pr.rows, dtype, pr.n, pr.d, &ix)) return rc;
      std::copy(pr.init_centroids, pr.init_centroids + pr.k * pr.d, centroids_out + co);
      const int rc = sc_kmeans_run(ix, pr.k, max_iter, mode, centroids_out + co, labels_out + lo,
                                   sizes_out + so, distortion_out + i, iters_out + i);
      sc_index_destroy(ix);
      if (rc) return rc;
      co += pr.k * pr.d;
      lo += pr.n;
      so += pr.k;
    }
    return SC_OK;
  }

  // ---- layout: one arena per buffer kind ----
  std::vector<KmProb> P(count);
  struct Off {
    int64_t rows, cent, lab, ps, pc, gs, gc, sum, cnt, x2, tab, c2f;
  };
  std::vector<Off> off(count);
  Off tot{};
  for (size_t i = 0; i < count; ++i) {
    const sc_kmeans_problem& pr = problems[i];
    KmProb& p = P[i];
    p.n = static_cast<int64_t>(pr.n);
    p.d = static_cast<int>(pr.d);
    p.ld = static_cast<int>(padded_dim(pr.d));
    p.k = static_cast<int>(pr.k);
    p.kpad = (p.k + 31) / 32 * 32;
    p.nb = (p.n + kBlockRows - 1) / kBlockRows;
    p.ng = (p.nb + kGroupBlocks - 1) / kGroupBlocks;
    const int64_t kd = static_cast<int64_t>(p.k) * std::max(p.d, 1);
    Off& o = off[i];
    o.rows = tot.rows;  tot.rows += p.n * p.ld;
    o.cent = tot.cent;  tot.cent += static_cast<int64_t>(p.k) * p.ld;
    o.lab = tot.lab;    tot.lab += p.n;
    o.ps = tot.ps;      tot.ps += p.nb * kd;
    o.pc = tot.pc;      tot.pc += p.nb * p.k;
    o.gs = tot.gs;      tot.gs += p.ng * kd;
    o.gc = tot.gc;      tot.gc += p.ng * p.k;
    o.sum = tot.sum;    tot.sum += kd;
    o.cnt = tot.cnt;    tot.cnt += p.k;
    o.x2 = tot.x2;      tot.x2 += p.nb + 2 * static_cast<int64_t>(p.k) + p.ld;
    o.tab = tot.tab;    tot.tab += static_cast<int64_t>(p.kpad) * p.ld;
    o.c2f = tot.c2f;    tot.c2f += p.kpad + 4;
  }
  DevBuf bP, bRows, bCent, bLab, bPs, bPc, bGs, bGc, bSum, bCnt, bX2, bHi, bMd, bLo, bC2f, bSt;
  SC_HIP(bP.alloc(sizeof(KmProb) * count, s));
  SC_HIP(bRows.alloc(sizeof(float) * tot.rows, s));
  SC_HIP(bCent.alloc(sizeof(double) * tot.cent, s));
  SC_HIP(bLab.alloc(sizeof(uint32_t) * tot.lab, s));
  SC_HIP(bPs.alloc(sizeof(double) * tot.ps, s));
  SC_HIP(bPc.alloc(sizeof(uint32_t) * tot.pc, s));
  SC_HIP(bGs.alloc(sizeof(double) * tot.gs, s));
  SC_HIP(bGc.alloc(sizeof(uint64_t) * tot.gc, s));
  SC_HIP(bSum.alloc(sizeof(double) * tot.sum, s));
  SC_HIP(bCnt.alloc(sizeof(uint64_t) * tot.cnt, s));
  SC_HIP(bX2.alloc(sizeof(double) * tot.x2, s));
  SC_HIP(bHi.alloc(sizeof(uint16_t) * tot.tab, s));
  SC_HIP(bMd.alloc(sizeof(uint16_t) * tot.tab, s));
  SC_HIP(bLo.alloc(sizeof(uint16_t) * tot.tab, s));
  SC_HIP(bC2f.alloc(sizeof(float) * tot.c2f, s));
  // per problem: state (32 B, 8-aligned) then the arrival counter
  const size_t st_stride = (sizeof(KmState) + 8 + 15) / 16 * 16;
  SC_HIP(bSt.alloc(st_stride * count, s));
  for (size_t i = 0; i < count; ++i) {
    KmProb& p = P[i];
    const Off& o = off[i];
    p.rows = bRows.as<float>() + o.rows;
    p.cent = bCent.as<double>() + o.cent;
    p.labels = bLab.as<uint32_t>() + o.lab;
    p.psum = bPs.as<double>() + o.ps;
    p.pcount = bPc.as<uint32_t>() + o.pc;
    p.gsum = bGs.as<double>() + o.gs;
    p.gcount = bGc.as<uint64_t>() + o.gc;
    p.sums = bSum.as<double>() + o.sum;
    p.counts = bCnt.as<uint64_t>() + o.cnt;
    p.x2block = bX2.as<double>() + o.x2;
    p.term = p.x2block + p.nb;
    p.c2d = p.term + p.k;
    p.mu = p.c2d + p.k;
    p.st = reinterpret_cast<KmState*>(bSt.as<char>() + st_stride * i);
    p.arrive = reinterpret_cast<uint32_t*>(bSt.as<char>() + st_stride * i + sizeof(KmState));
    p.bhi = bHi.as<uint16_t>() + o.tab;
    p.bmd = bMd.as<uint16_t>() + o.tab;
    p.blo = bLo.as<uint16_t>() + o.tab;
    p.c2f = bC2f.as<float>() + o.c2f;
    p.cmax = p.c2f + p.kpad;
  }
  // Two streams from here on: cs carries every host-to-device copy, s every
  // kernel.  The problems go in groups of consecutive problems with about
  // equal row bytes; a group's iterations run on s while the next group's
  // rows go up on cs (the copy engines need none of the CUs that the
  // persistent label launches hold), and s waits for a group's rows
  // through an event.
  hipStream_t cs = copy_stream_for_device(dev);
  if (!cs) return fail(SC_ERR_DEVICE, "no copy stream for the device");
  std::vector<std::unique_ptr<Group>> groups;
  DevBuf bItems;
  struct Events {
    std::vector<hipEvent_t> e;
    ~Events() {
      for (hipEvent_t x : e) (void)hipEventDestroy(x);
    }
    hipError_t add(hipEvent_t* out) {
      hipEvent_t x = nullptr;
      const hipError_t r = hipEventCreateWithFlags(&x, hipEventDisableTiming);
      if (r == hipSuccess) {
        e.push_back(x);
        *out = x;
      }
      return r;
    }
  } evs;
  // Declared after every buffer that cs writes: whatever the return, both
  // streams are drained before those buffers are released.
  struct Drain {
    hipStream_t a, b;
    ~Drain() {
      (void)hipStreamSynchronize(a);
      (void)hipStreamSynchronize(b);
    }
  } drain{s, cs};
  hipEvent_t allocated = nullptr;
  SC_HIP(evs.add(&allocated));
  SC_HIP(hipEventRecord(allocated, s));
  SC_HIP(hipStreamWaitEvent(cs, allocated, 0));
  if (int rc = upload_staged(bP.p, P.data(), sizeof(KmProb) * count, cs)) return rc;
  // the initial centroids of every problem, padded on the host, in one copy
  std::vector<double> hcent0(static_cast<size_t>(tot.cent), 0.0);
  for (size_t i = 0; i < count; ++i) {
    const sc_kmeans_problem& pr = problems[i];
    for (size_t c = 0; c < pr.k; ++c)
      std::copy(pr.init_centroids + c * pr.d, pr.init_centroids + (c + 1) * pr.d,
                hcent0.data() + off[i].cent + c * P[i].ld);
  }
  if (int rc = upload_staged(bCent.p, hcent0.data(), sizeof(double) * tot.cent, cs)) return rc;
  const KmProb* dP = bP.as<KmProb>();

  // ---- groups: cut where the running row bytes pass g / ngroups ----
  {
    const int64_t row_bytes = static_cast<int64_t>(sizeof(float)) * tot.rows;
    const int64_t ng = std::max<int64_t>(1, std::min<int64_t>(kUploadGroups, row_bytes / kUploadGroupBytes));
    int64_t acc = 0;
    size_t first = 0;
    for (size_t i = 0; i < count; ++i) {
      acc += static_cast<int64_t>(sizeof(float)) * P[i].n * P[i].ld;
      if (i + 1 == count || acc * ng >= row_bytes * static_cast<int64_t>(groups.size() + 1)) {
        auto g = std::make_unique<Group>();
        g->first = first;
        g->count = i + 1 - first;
        groups.push_back(std::move(g));
        first = i + 1;
      }
    }
  }

  // ---- items of every group (problem indices relative to the group):
  // sums items over every block, label items per shape class; one copy ----
  std::vector<uint2> hitems;
  for (auto& gp : groups) {
    Group& G = *gp;
    const KmProb* HP = P.data() + G.first;
    int64_t maxnb = 0;
    for (size_t i = 0; i < G.count; ++i) {
      maxnb = std::max(maxnb, HP[i].nb);
      G.ldmax = std::max(G.ldmax, HP[i].ld);
      G.rows += HP[i].n;
    }
    // block-major across problems so concurrent workgroups spread over problems
    for (int64_t b = 0; b < maxnb; ++b)
      for (size_t i = 0; i < G.count; ++i) {
        const KmProb& p = HP[i];
        if (b >= p.nb) continue;
        G.all.push_back(make_uint2(static_cast<unsigned>(i), static_cast<unsigned>(b)));
        const int kbm = kbm_of(p.k), ksm = ksm_of(p.ld);
        const bool exact = (p.k + 31) / 32 == kbm && p.ld / 16 == ksm;
        Klass& K = G.klass[(kbm * 16 + ksm) * 2 + (exact ? 1 : 0)];
        K.kbm = kbm;
        K.ksm = ksm;
        K.exact = exact;
        K.kmax = std::max(K.kmax, p.k);
        K.ldmax = std::max(K.ldmax, p.ld);
        // the label segments of this block
        const int64_t seg_end = std::min<int64_t>((b + 1) * (kBlockRows / kSegRows),
                                                  (p.n + kSegRows - 1) / kSegRows);
        for (int64_t sg = b * (kBlockRows / kSegRows); sg < seg_end; ++sg)
          K.items.push_back(make_uint2(static_cast<unsigned>(i), static_cast<unsigned>(sg)));
      }
    G.all_at = hitems.size();
    hitems.insert(hitems.end(), G.all.begin(), G.all.end());
    for (auto& kv : G.klass) {
      kv.second.at = hitems.size();
      hitems.insert(hitems.end(), kv.second.items.begin(), kv.second.items.end());
    }
    if (int rc = G.red.build(HP, G.count, cs)) return rc;
  }
  SC_HIP(bItems.alloc(sizeof(uint2) * hitems.size(), cs));
  if (int rc = upload_staged(bItems.p, hitems.data(), sizeof(uint2) * hitems.size(), cs)) return rc;

  const int cus = device_cus();

  for (auto& gp : groups) {
    Group& G = *gp;
    // the group's rows: one staged stream, padded on the host
    {
      std::vector<StageSeg> segs(G.count);
      for (size_t i = 0; i < G.count; ++i) {
        const size_t pi = G.first + i;
        segs[i] = StageSeg{problems[pi].rows, problems[pi].n, problems[pi].d * sizeof(float),
                           static_cast<size_t>(P[pi].ld) * sizeof(float)};
      }
      if (int rc = upload_staged_segments(bRows.as<float>() + off[G.first].rows, segs.data(),
                                          G.count, cs))
        return rc;
    }
    hipEvent_t up = nullptr;
    SC_HIP(evs.add(&up));
    SC_HIP(hipEventRecord(up, cs));
    SC_HIP(hipStreamWaitEvent(s, up, 0));

    const KmProb* dG = dP + G.first;
    const uint2* d_all = bItems.as<uint2>() + G.all_at;
    const int64_t nall = static_cast<int64_t>(G.all.size());
    const int gc = static_cast<int>(G.count);
    const unsigned cgrid = static_cast<unsigned>((G.count + 255) / 256);
    hipLaunchKernelGGL(kmb_init_kernel, dim3(cgrid), dim3(256), 0, s, dG, gc);
    hipLaunchKernelGGL(kmb_mu_kernel, dim3(static_cast<unsigned>(gc)), dim3(128), 0, s, dG, gc);
    hipLaunchKernelGGL(kmb_x2_kernel, dim3(1024), dim3(NT), 0, s, dG, d_all, nall);
    hipLaunchKernelGGL(kmb_x2_total_kernel, dim3(cgrid), dim3(256), 0, s, dG, gc);
    SC_HIP(hipGetLastError());
    if (int rc = kmeans_tables_launch(dG, G.count, s)) return rc;

    // The shape classes' label launches go one after another on s, the
    // most work first (items x k blocks x row blocks): each launch is
    // persistent over the whole chip, and the small classes at the end
    // leave short tails.  (One side stream per class, forked and joined in
    // every iteration, ran slower: the branches share the process's four
    // hardware queues, so they queued behind one another anyway.)
    std::vector<const Klass*> order;
    for (auto& kv : G.klass) order.push_back(&kv.second);
    auto work = [](const Klass* K) {
      return static_cast<double>(K->items.size()) * K->kbm * K->ksm;
    };
    std::stable_sort(order.begin(), order.end(),
                     [&](const Klass* a, const Klass* b) { return work(a) > work(b); });
    auto iteration = [&](int mult) -> int {
      for (const Klass* K : order)
        if (int rc = launch_label(K->kbm, K->ksm, mult, dG, bItems.as<uint2>() + K->at,
                                  static_cast<int64_t>(K->items.size()), K->exact, cus, s))
          return rc;
      if (int rc = launch_sums<float>(dG, d_all, nall, G.ldmax, kSumMaxK, cus, s)) return rc;
      return kmeans_reduce_launch(dG, G.red, true, true, s);
    };

    // ---- launch shape: cached, or timed on the first iterations ----
    // Candidates: label workgroups per CU (1, 2, 3, 4, 6, 8; four waves
    // each).  Every shape gives the same labels and sums (the sums' order is
    // fixed per block), so the timed iterations are real ones.
    std::vector<int64_t> key;
    for (auto& kv : G.klass) {
      key.push_back(kv.first);
      key.push_back(static_cast<int64_t>(kv.second.items.size()));
    }
    {
      std::lock_guard<std::mutex> lk(g_tune_mu);
      for (auto& e : g_tune)
        if (e.key == key) {
          G.waves = e.waves;
          G.mult = e.mult;
        }
    }
    size_t it_done = 0;
    if (G.mult == 0) {
      const int cand[6][2] = {{4, 1}, {4, 2}, {4, 3}, {4, 4}, {4, 6}, {4, 8}};
      float best = 1e30f;
      struct TimerPair {
        hipEvent_t a = nullptr, b = nullptr;
        ~TimerPair() {
          if (a) (void)hipEventDestroy(a);
          if (b) (void)hipEventDestroy(b);
        }
      } tp;
      SC_HIP(hipEventCreate(&tp.a));
      SC_HIP(hipEventCreate(&tp.b));
      for (int c = 0; c < 6 && it_done < max_iter; ++c) {
        SC_HIP(hipEventRecord(tp.a, s));
        if (int rc = iteration(cand[c][1])) return rc;
        SC_HIP(hipEventRecord(tp.b, s));
        SC_HIP(hipEventSynchronize(tp.b));
        float ms = 0.0f;
        SC_HIP(hipEventElapsedTime(&ms, tp.a, tp.b));
        ++it_done;
        if (ms < best) {
          best = ms;
          G.waves = cand[c][0];
          G.mult = cand[c][1];
        }
      }
      if (it_done == 6) {  // a full comparison: kept for later calls
        std::lock_guard<std::mutex> lk(g_tune_mu);
        g_tune.push_back(TuneEntry{key, G.waves, G.mult});
      }
    }
    // ---- remaining iterations as one graph, launched without waiting ----
    if (it_done < max_iter) {
      ProfScope ps("kmeans_batch", s);
      hipGraph_t graph = nullptr;
      hipGraphExec_t exec = nullptr;
      SC_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
      int crc = SC_OK;
      for (size_t it = it_done; it < max_iter && crc == SC_OK; ++it) crc = iteration(G.mult);
      hipError_t ce = hipStreamEndCapture(s, &graph);
      if (crc) {
        if (graph) (void)hipGraphDestroy(graph);
        return crc;
      }
      if (ce != hipSuccess) return hip_fail(ce, "hipStreamEndCapture");
      ce = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
      if (ce != hipSuccess) {
        (void)hipGraphDestroy(graph);
        return hip_fail(ce, "hipGraphInstantiate");
      }
      // kept by the group until both streams are drained
      G.graph = graph;
      G.exec = exec;
      ce = hipGraphLaunch(exec, s);
      if (ce != hipSuccess) return hip_fail(ce, "hipGraphLaunch");
    }
  }
  SC_HIP(hipStreamSynchronize(s));
  // ---- results ----
  // the states sit st_stride apart in one arena: one copy for all
  std::vector<char> hst(st_stride * count);
  if (int rc = download_staged(hst.data(), bSt.p, st_stride * count, s)) return rc;
  std::vector<KmState> hs(count);
  for (size_t i = 0; i < count; ++i) std::memcpy(&hs[i], hst.data() + st_stride * i, sizeof(KmState));
  // the label and size arenas hold the problems in order, like the outputs;
  // the centroid arena is copied whole and its row padding dropped here
  if (int rc = download_staged(labels_out, bLab.p, sizeof(uint32_t) * tot.lab, s)) return rc;
  if (int rc = download_staged(sizes_out, bCnt.p, sizeof(uint64_t) * tot.cnt, s)) return rc;
  std::vector<double> hcent(static_cast<size_t>(tot.cent));
  if (int rc = download_staged(hcent.data(), bCent.p, sizeof(double) * tot.cent, s)) return rc;
  SC_HIP(hipStreamSynchronize(s));
  size_t co = 0;
  for (size_t i = 0; i < count; ++i) {
    const KmProb& p = P[i];
    const double* src = hcent.data() + off[i].cent;
    for (int c = 0; c < p.k; ++c)
      std::copy(src + static_cast<size_t>(c) * p.ld, src + static_cast<size_t>(c) * p.ld + p.d,
                centroids_out + co + static_cast<size_t>(c) * p.d);
    co += static_cast<size_t>(p.k) * p.d;
  }
  uint64_t fb = 0;
  for (size_t i = 0; i < count; ++i) {
    distortion_out[i] = hs[i].distortion;
    iters_out[i] = hs[i].iters;
    fb += hs[i].fallback;
  }
  // the launch shape reported is the one of the group with the most rows
  const Group* big = groups.front().get();
  for (auto& gp : groups)
    if (gp->rows > big->rows) big = gp.get();
  sc_stats& st = last_stats();
  st = sc_stats{};
  st.queries = count;
  st.uncertified = fb;
  st.launch_waves = static_cast<uint64_t>(big->waves);
  st.launch_groups_per_cu = static_cast<uint64_t>(big->mult);
  st.upload_groups = groups.size();
  return SC_OK;
}
