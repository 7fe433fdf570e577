// perm_impl.hpp -- Glynn / BB-FG Gray-code permanent on gfx950 (fp64, kappa, dd).
//
// Algorithm (reference: core/permanent.cu:30-76, cpu_ref/permanent.py:108-139):
//   perm(A) = 2^-(n-1) sum_{delta, delta_0=+1} (prod_k delta_k) prod_r sum_c delta_c A[r,c]
// walked in reflected Gray-code order, so consecutive terms differ in one
// delta_col and the row sums change by +-2 A[:,col].
//
// MI355X mapping (this file's own design, not the reference's one-thread-per-
// matrix): the 2^(n-1) term space of one matrix is cut into contiguous,
// 2^M-aligned Gray ranges, one per lane; for large n the ranges of one matrix
// also span several workgroups ("chunks"; 2^M comes from a per-size table,
// perm_tune.hpp). Because every range starts at a
// multiple of 2^M, the flipped column ctz(i) of a lane's j-th step is ctz(j) for
// ALL lanes: the whole wave walks the same column sequence in lockstep. The row
// sums live in VGPRs (fully unrolled over a compile-time n); columns 1..HOT
// (flipped every 2nd, 4th, ... step) are cached in VGPRs, the rarer columns are
// read from an LDS copy of A^T with a wave-uniform address (a broadcast read).
// Lane partials are combined by a butterfly over the group's lanes, chunk
// partials by a fixed-order second pass. The chunking depends only on n and
// the tier family, so a matrix's value never depends on what else is in the
// batch.
#pragma once

#include <limits.h>

#include "cert.hpp"
#include "common.hpp"
#include "perm.hpp"

namespace gbsk {

// rounding depth of the certificate arithmetic (cert.hpp): per lane 8 * 2^M + 16 N,
// plus the butterfly and the chunk sum
__device__ inline double perm_cert_depth(int N, int M, int W) {
  return 8.0 * (double)(1u << M) + 16.0 * N + 4.0 * W + 64.0;
}

// Per-lane Gray range [start, start + 2^M): initial row sums at gray(start),
// then 2^M - 1 single-column updates. Returns the signed, unscaled partial.
// Shared by the fp64 plain and kappa modes (identical value arithmetic).
// CERT: also carry a running bound (1-norm, round-to-nearest with a final
// inflation, see cert.hpp) of |value - exact|: er[r] for the row sums, ep for a
// product, E for the lane's partial.
template <int N, int HOT, bool KAPPA, bool CERT>
__device__ inline void glynn_range_fp64(const cplx* __restrict__ AT,  // LDS, AT[c*N + r]
                                        uint32_t start, int M, cplx& acc_out, double& abs_out) {
  cplx rs[N];
  double er[N];
  const uint32_t g = start ^ (start >> 1);
#pragma unroll
  for (int r = 0; r < N; ++r) {
    rs[r] = AT[r];  // column 0, delta_0 = +1 (exact)
    er[r] = 0.0;
  }
#pragma unroll 1
  for (int c = 1; c < N; ++c) {
    const double s = ((g >> (c - 1)) & 1u) ? -1.0 : 1.0;
#pragma unroll
    for (int r = 0; r < N; ++r) {
      rs[r] = c_axpy(s, AT[c * N + r], rs[r]);
      if (CERT) er[r] = cert_round(rs[r], er[r]);
    }
  }
  // hot columns: 1..HOT
  cplx hot[HOT > 0 ? HOT : 1][N];
#pragma unroll
  for (int h = 0; h < HOT; ++h)
#pragma unroll
    for (int r = 0; r < N; ++r) hot[h][r] = AT[(h + 1) * N + r];

  double ep = 0.0;  // bound of the last product (CERT)
  auto product = [&]() {
    // four interleaved chains (rows r = q mod 4), then (t0 t1)(t2 t3): fixed order
    cplx t[4];
    double et[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      t[q] = q < N ? rs[q] : cplx{1.0, 0.0};
      et[q] = q < N ? er[q] : 0.0;
    }
#pragma unroll
    for (int r = 4; r < N; ++r) {
      if (CERT) et[r & 3] = cert_mul(t[r & 3], et[r & 3], rs[r], er[r]);
      t[r & 3] = c_mul(t[r & 3], rs[r]);
    }
    if constexpr (N == 1) {
      ep = et[0];
      return t[0];
    }
    if constexpr (N == 2) {
      if (CERT) ep = cert_mul(t[0], et[0], t[1], et[1]);
      return c_mul(t[0], t[1]);
    }
    if constexpr (N == 3) {
      const cplx t01 = c_mul(t[0], t[1]);
      if (CERT) ep = cert_mul(t01, cert_mul(t[0], et[0], t[1], et[1]), t[2], et[2]);
      return c_mul(t01, t[2]);
    }
    const cplx t01 = c_mul(t[0], t[1]), t23 = c_mul(t[2], t[3]);
    if (CERT) ep = cert_mul(t01, cert_mul(t[0], et[0], t[1], et[1]), t23, cert_mul(t[2], et[2], t[3], et[3]));
    return c_mul(t01, t23);
  };

  cplx acc = product();  // term j = 0: start is even, sign +
  double aacc = KAPPA ? c_abs(acc) : 0.0;
  double E = CERT ? ep : 0.0;
  const uint32_t nsteps = 1u << M;
  constexpr int U = HOT;  // static block length 2^U: steps t = 1..2^U-1 use hot columns
  if constexpr (U == 0) {
    for (uint32_t j = 1; j < nsteps; ++j) {
      const int k = __builtin_ctz(j);
      const uint32_t i = start + j;
      const double step = ((i >> (k + 1)) & 1u) ? 2.0 : -2.0;
      const cplx* col = AT + (k + 1) * N;
#pragma unroll
      for (int r = 0; r < N; ++r) {
        rs[r] = c_axpy(step, col[r], rs[r]);
        if (CERT) er[r] = cert_round(rs[r], er[r]);
      }
      cplx p = product();
      acc = (j & 1u) ? c_sub(acc, p) : c_add(acc, p);
      if (KAPPA) aacc += c_abs(p);
      if (CERT) E = cert_round(acc, E + ep);
    }
  } else {
    // blocks of 2^U steps: steps t < 2^U flip hot column ctz(t) + 1, step 2^U a
    // cold column. The last block stops before its cold step (j = 2^M lies
    // outside the range); it is peeled so that the loop body has no exit test
    // (a data-dependent break there cost ~60 registers and half the occupancy)
    const uint32_t nblocks = nsteps >> U;  // >= 1: M >= U
    auto body = [&](uint32_t jb, int t) __attribute__((always_inline)) {
        const uint32_t j = (jb << U) + (uint32_t)t;
        const uint32_t i = start + j;
        int k;
        if (t < (1 << U)) {
          k = __builtin_ctz((unsigned)t);
        } else {
          k = __builtin_ctz(j);
        }
        const double step = ((i >> (k + 1)) & 1u) ? 2.0 : -2.0;
        if (t < (1 << U)) {
#pragma unroll
          for (int r = 0; r < N; ++r) rs[r] = c_axpy(step, hot[__builtin_ctz((unsigned)t)][r], rs[r]);
        } else {
          const cplx* col = AT + (k + 1) * N;
#pragma unroll
          for (int r = 0; r < N; ++r) rs[r] = c_axpy(step, col[r], rs[r]);
        }
        if (CERT) {
#pragma unroll
          for (int r = 0; r < N; ++r) er[r] = cert_round(rs[r], er[r]);
        }
        cplx p = product();
        acc = (t & 1) ? c_sub(acc, p) : c_add(acc, p);
        if (KAPPA) aacc += c_abs(p);
        if (CERT) E = cert_round(acc, E + ep);
    };
    for (uint32_t jb = 0; jb + 1 < nblocks; ++jb) {
#pragma unroll
      for (int t = 1; t <= (1 << U); ++t) body(jb, t);
    }
#pragma unroll
    for (int t = 1; t < (1 << U); ++t) body(nblocks - 1, t);
  }
  acc_out = acc;
  abs_out = CERT ? E : aacc;
}

// Double-double row sums. Every entry is split once, per row and component, on
// a grid g = 2^(k - 53) with 2^k > sum_c |a_rc|: a = hi + lo exactly, hi = g rint(a / g),
// |lo| <= g / 2. Any sum of +-hi is a multiple of g below 2^53 g, so it is exact in
// binary64, and a Gray step is one fma each for the high and the low sums (4 a
// row; a double-double addition of 2a took 22 operations). The low sums round at
// most at u |lo| <= u n g / 2, a double-double addition's own rounding, and not
// at all where the row's entries lie within a few binary orders of one another
// (lo is then a handful of bits). The walk hands FastTwoSum(hi, lo) to the
// products, which is exact: hi is a multiple of ulp(lo).
struct RowSplit {
  int k;  // exponent; INT_MIN: nothing to split (zero, infinite or NaN row)
  __device__ static RowSplit of(double sum) {
    // frexp's exponent: 2^k > sum (one instruction, subnormal numbers too)
    return RowSplit{sum > 0.0 && sum < INFINITY
                        ? __builtin_amdgcn_frexp_exp(fmin(sum * (1.0 + 0x1p-40), 1.79769313486231570e308))
                        : INT_MIN};
  }
  __device__ double hi(double a) const { return k == INT_MIN ? a : ldexp(rint(ldexp(a, 53 - k)), k - 53); }
  // The low sums do not round either if the smallest nonzero entry, whose frexp
  // exponent is `least`, is not far below: low parts are multiples of 2^(least - 53)
  // and n of them, at most 2^(k - 54) each, stay below 2^53 of those (n <= 2^5).
  __device__ bool exact(int least) const { return k == INT_MIN || k - 49 <= least; }
};
// min(least, frexp exponent of a), a nonzero
__device__ __forceinline__ int min_exp(double a, int least) {
  const int e = __builtin_amdgcn_frexp_exp(a);
  return a != 0.0 && e < least ? e : least;
}

// split the `mats` staged matrices in place: AT keeps the high parts, AL gets the
// low; inexact[q] (CERT): a low sum of matrix q may round
template <int N, int MPW, bool CERT>
__device__ inline void split_rows(cplx (&AT)[MPW][N * N], cplx (&AL)[MPW][N * N], int mats, int (&inexact)[MPW]) {
  static_assert(N <= 32, "RowSplit::exact");
  if constexpr (CERT) {
    for (int q = threadIdx.x; q < MPW; q += 64) inexact[q] = 0;
    __syncthreads();
  }
  for (int t = threadIdx.x; t < mats * N * 2; t += 64) {  // (matrix, row, component)
    const int q = t / (2 * N), r = (t >> 1) % N;
    double* const a = reinterpret_cast<double*>(&AT[q][r]) + (t & 1);
    double* const l = reinterpret_cast<double*>(&AL[q][r]) + (t & 1);
    double sum = 0.0;
    int least = INT_MAX;
#pragma unroll 4
    for (int c = 0; c < N; ++c) {
      sum += fabs(a[2 * c * N]);
      if constexpr (CERT) least = min_exp(a[2 * c * N], least);
    }
    const RowSplit s = RowSplit::of(sum);
    if (CERT && !s.exact(least)) inexact[q] = 1;
#pragma unroll 4
    for (int c = 0; c < N; ++c) {
      const double v = a[2 * c * N], h = s.hi(v);
      a[2 * c * N] = h;
      l[2 * c * N] = s.k == INT_MIN ? 0.0 : v - h;
    }
  }
  __syncthreads();
}

// Up to this side a lane splits its own copy of the matrix in registers and its few
// terms are unrolled (2^M is 2^MLIM there whatever the table says): the pass over
// LDS and its barrier took longer than the additions it saves. dd, B = 200000: n = 2 / 3 / 4
// 5.0 / 12.5 / 28.5 us with double-double additions, 6.2 / 15.1 / 34.9 split in LDS, 5.3 / 10.6 / 23.0 here.
constexpr int PERM_DD_REG = 4;
template <int N>
__device__ __forceinline__ bool split_own(const cplx* A, cplx (&H)[N * N], cplx (&L)[N * N]) {
  bool exact = true;  // no low sum rounds
#pragma unroll
  for (int r = 0; r < N; ++r) {
    double sr = 0.0, si = 0.0;
    int lr = INT_MAX, li = INT_MAX;
#pragma unroll
    for (int c = 0; c < N; ++c) {
      H[c * N + r] = A[c * N + r];
      sr += fabs(H[c * N + r].re);
      si += fabs(H[c * N + r].im);
      lr = min_exp(H[c * N + r].re, lr);
      li = min_exp(H[c * N + r].im, li);
    }
    const RowSplit kr = RowSplit::of(sr), ki = RowSplit::of(si);
    exact = exact && kr.exact(lr) && ki.exact(li);
#pragma unroll
    for (int c = 0; c < N; ++c) {
      const cplx a = H[c * N + r], h{kr.hi(a.re), ki.hi(a.im)};
      H[c * N + r] = h;
      L[c * N + r] = cplx{kr.k == INT_MIN ? 0.0 : a.re - h.re, ki.k == INT_MIN ? 0.0 : a.im - h.im};
    }
  }
  return exact;
}

// one row's sum as a normalised double-double
__device__ inline ddc row_sum(cplx h, cplx l) { return ddc{fast_two_sum(h.re, l.re), fast_two_sum(h.im, l.im)}; }

// f(1), ..., f(e - 1); small sides unrolled, e = E there
template <int N, int E, class F>
__device__ __forceinline__ void perm_dd_terms(uint32_t e, const F& f) {
  if constexpr (N <= PERM_DD_REG) {
    static_assert(PermCfg<N, 1>::MLIM <= 2, "no entry below 2^2 terms a lane: M is MLIM");
#pragma unroll
    for (uint32_t j = 1; j < (uint32_t)E; ++j) f(j);
  } else {
    for (uint32_t j = 1; j < e; ++j) f(j);
  }
}
template <int N, class F>
__device__ __forceinline__ void perm_dd_columns(const F& f) {
  if constexpr (N <= PERM_DD_REG) {
#pragma unroll
    for (int c = 1; c < N; ++c) f(c);
  } else {
#pragma unroll 1
    for (int c = 1; c < N; ++c) f(c);
  }
}

// Same walk in complex double-double (reference: core/permanent_dd.cu:34-73,
// cpu_ref/permanent.py:142-189). What bounds it: FP64 issue, 842 operations
// a term at n = 16 (16 rows at 10, 15 products at 44), 81% of the nominal rate. Measured on MI355X,
// double-double additions and separately normalised products -> this: n = 8 / 12 /
// 16 / 20 (B = 16384 / 16384 / 16384 / 238) 66 / 1066 / 18381 / 5501 -> 47 / 805 / 14159 /
// 4086 us, certified n = 16 (B = 1907) 5549 -> 3139 us; values the same binary64 bits.
template <int N>
__device__ __forceinline__ void glynn_range_dd(const cplx* AT, const cplx* AL, uint32_t start, int M, ddc& acc_out) {
  cplx rh[N], rl[N];
  const uint32_t g = start ^ (start >> 1);
#pragma unroll
  for (int r = 0; r < N; ++r) {
    rh[r] = AT[r];
    rl[r] = AL[r];
  }
  auto update = [&](double s, int c) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < N; ++r) {
      rh[r] = c_axpy(s, AT[c * N + r], rh[r]);
      rl[r] = c_axpy(s, AL[c * N + r], rl[r]);
    }
  };
  auto first = [&](int c) __attribute__((always_inline)) { update(((g >> (c - 1)) & 1u) ? -1.0 : 1.0, c); };
  perm_dd_columns<N>(first);
  auto product = [&]() {
    // two interleaved chains (even / odd rows), then their product
    ddc t0 = row_sum(rh[0], rl[0]);
#pragma unroll
    for (int r = 2; r < N; r += 2) t0 = ddc_mul(t0, row_sum(rh[r], rl[r]));
    if constexpr (N == 1) return t0;
    ddc t1 = row_sum(rh[1], rl[1]);
#pragma unroll
    for (int r = 3; r < N; r += 2) t1 = ddc_mul(t1, row_sum(rh[r], rl[r]));
    return ddc_mul(t0, t1);
  };
  ddc acc = product();
  auto term = [&](uint32_t j) __attribute__((always_inline)) {
    const int k = __builtin_ctz(j);
    const uint32_t i = start + j;
    update(((i >> (k + 1)) & 1u) ? 2.0 : -2.0, k + 1);
    ddc p = product();
    acc = (j & 1u) ? ddc_sub(acc, p) : ddc_add(acc, p);
  };
  perm_dd_terms<N, 1 << PermCfg<N, 1>::MLIM>(1u << M, term);
  acc_out = acc;
}

// Compiler barrier on a bound accumulator (emits no instruction). Without it
// LLVM sinks each operation's error computation to where the bound is next
// read, keeping three intermediates per row sum alive across the whole step:
// the certified-dd walk then spilled 900-1800 VGPRs to scratch (40-120x the dd
// walk's time); with it the bound is folded in as the values are formed.
__device__ __forceinline__ void pin(double& v) { asm volatile("" : "+v"(v)); }

// glynn_range_dd with a running bound (certified double-double). The values
// are glynn_range_dd's bit for bit. E bounds the error of every row sum: zero where
// neither high nor low sums round (exact, RowSplit), which entries within 2^49 of
// their row's sum ensure; else each step adds the largest of the N low sums'
// roundings, u |low sum| (so charged for every matrix, bounds of cancelling inputs
// were 1.9, 2.6 and 9 times as wide as with double-double additions at n = 16, 17 and
// 22; with rows that span 24 decades they are 1.2, 1.9 and 3.6 times at n = 6, 10 and 22.
// The errors themselves, by TwoSum, take these away but cost 1.12-1.43 times the time,
// in a branch of their own 1.15-1.2 times from n = 15 on, in registers). Products and the signed
// accumulation propagate it with the 1-norm product rule plus each operation's own error.
template <int N>
__device__ __forceinline__ void glynn_range_ddcert(const cplx* AT, const cplx* AL, uint32_t start, int M, bool exact,
                                                   ddc& acc_out, double& e_out) {
  cplx rh[N], rl[N];
  const uint32_t g = start ^ (start >> 1);
  const double eu = exact ? 0.0 : CERT_U, ef = exact ? 0.0 : CERT_UFL;
  double E = 0.0;
#pragma unroll
  for (int r = 0; r < N; ++r) {
    rh[r] = AT[r];
    rl[r] = AL[r];
  }
  auto update = [&](double s, int c) __attribute__((always_inline)) {
    double m = 0.0;
#pragma unroll
    for (int r = 0; r < N; ++r) {
      rh[r] = c_axpy(s, AT[c * N + r], rh[r]);
      rl[r] = c_axpy(s, AL[c * N + r], rl[r]);
      m = fmax(m, cert_norm1(rl[r]));
      // every fifth row: the next rows' loads then pass the barrier; at every row
      // n = 21 / 24 / 26 (B = 256 / 64 / 16) took 22.7 / 51.5 / 60.2 ms, so 19.0 / 43.8 / 49.6
      if (r % 5 == 4) pin(m);
    }
    E += fma(eu, m, ef);
  };
  auto first = [&](int c) __attribute__((always_inline)) { update(((g >> (c - 1)) & 1u) ? -1.0 : 1.0, c); };
  perm_dd_columns<N>(first);
  auto product = [&](double& ep) {
    ddc t0 = row_sum(rh[0], rl[0]);
    double e0 = E;
#pragma unroll
    for (int r = 2; r < N; r += 2) {
      double eo;
      const ddc rs = row_sum(rh[r], rl[r]);
      const ddc t = cddc_mul(t0, rs, &eo);
      e0 = cddc_mul_bound(t0, e0, rs, E, eo);
      pin(e0);
      t0 = t;
    }
    if constexpr (N == 1) {
      ep = e0;
      return t0;
    }
    ddc t1 = row_sum(rh[1], rl[1]);
    double e1 = E;
#pragma unroll
    for (int r = 3; r < N; r += 2) {
      double eo;
      const ddc rs = row_sum(rh[r], rl[r]);
      const ddc t = cddc_mul(t1, rs, &eo);
      e1 = cddc_mul_bound(t1, e1, rs, E, eo);
      pin(e1);
      t1 = t;
    }
    double eo;
    const ddc t = cddc_mul(t0, t1, &eo);
    ep = cddc_mul_bound(t0, e0, t1, e1, eo);
    return t;
  };
  double ea;
  ddc acc = product(ea);
  auto term = [&](uint32_t j) __attribute__((always_inline)) {
    const int k = __builtin_ctz(j);
    const uint32_t i = start + j;
    update(((i >> (k + 1)) & 1u) ? 2.0 : -2.0, k + 1);
    double ep, eo;
    const ddc p = product(ep);
    acc = (j & 1u) ? cddc_sub(acc, p, &eo) : cddc_add(acc, p, &eo);
    ea = ea + ep + eo;
  };
  perm_dd_terms<N, 1 << PermCfg<N, 1>::MLIM>(1u << M, term);
  acc_out = acc;
  e_out = ea;
}

// butterfly sum over G lanes of (ddc value, bound): group_sum<G>(ddc)'s order
template <int G>
__device__ inline void cddc_group_sum(ddc& v, double& e) {
#pragma unroll
  for (int m = 1; m < G; m <<= 1) {
    ddc o;
    o.re.hi = shfl_xor_d(v.re.hi, m);
    o.re.lo = shfl_xor_d(v.re.lo, m);
    o.im.hi = shfl_xor_d(v.im.hi, m);
    o.im.lo = shfl_xor_d(v.im.lo, m);
    const double eo = shfl_xor_d(e, m);
    const bool low = (threadIdx.x & m) == 0;
    double r;
    v = low ? cddc_add(v, o, &r) : cddc_add(o, v, &r);
    e = e + eo + r;
  }
}

// rounding depth of the certified-dd bound: the row bound's 2^M-step
// accumulation, the product chains, the butterfly and the chunk sum
__device__ inline double perm_ddcert_depth(int N, int M, int W) {
  return 8.0 * (double)(1u << M) + 16.0 * N + 8.0 * W + 128.0;
}

// One workgroup = one wave = MPW matrices x LPM lanes (or one chunk of one
// matrix when the matrix is split over W workgroups).
//   out      : final values (W == 1) or chunk partials [B][W] (W > 1)
//   aux      : kappa sum|term| (final or partial), may be null in plain mode
//   M, W     : the run-time split (log2 terms per lane, workgroups per matrix)
// fp64, kappa and dd ask for at least two waves per SIMD: without the hint the
// fp64 kernel takes 256 VGPRs plus a few AGPRs at n = 15..25 (one wave per
// SIMD); with it n = 14..18 fit in 202..250 VGPRs and n = 19..25 spill 1..6
// VGPRs. The certified modes carry a bound per row sum and would spill dozens
// of VGPRs to scratch: they keep one wave per SIMD and AGPR spill space.
template <int MODE>
constexpr int perm_min_waves() { return (MODE == PERM_CERT || MODE == PERM_DDCERT) ? 1 : 2; }

// complex numbers of LDS one workgroup uses: the matrices (dd: high, then low parts)
template <int N, int MODE>
constexpr int perm_lds() {
  return (64 / PermCfg<N, perm_is_dd(MODE) ? 1 : 0>::LPM) * N * N * (perm_is_dd(MODE) && N > PERM_DD_REG ? 2 : 1);
}

template <int N, int MODE>
__device__ __forceinline__ void perm_workgroup(const cplx* __restrict__ mats, int B, cplx* __restrict__ out,
                                               double* __restrict__ aux, int g8, int M, int W, int64_t wg,
                                               cplx* lds) {
  using C = PermCfg<N, perm_is_dd(MODE) ? 1 : 0>;
  constexpr int LPM = C::LPM, MPW = 64 / LPM;
  cplx(&AT)[MPW][N * N] = *reinterpret_cast<cplx(*)[MPW][N * N]>(lds);
  const int lane = threadIdx.x;
  const int gidx = lane / LPM, sub = lane % LPM;
  // workgroup -> (matrix group, chunk). Workgroups are dealt to the 8 XCDs in
  // id order, so for a split matrix (W > 1) the id is decoded such that all W
  // chunks of one group share an XCD (its L2 then fetches the matrix once).
  int64_t grp;
  int chunk;
  if (W == 1) {
    grp = wg;
    chunk = 0;
  } else {
    // g8 = min(8, groups): with fewer than 8 groups no padding workgroups
    const int64_t k = wg / g8;
    grp = (k / W) * g8 + wg % g8;
    chunk = (int)(k % W);
  }
  const int64_t mat0 = grp * MPW;
  if (mat0 >= B) return;  // padding workgroup (uniform exit, before any barrier)
  // stage MPW matrices transposed into LDS
  // (eight loads in flight a lane: one at a time cost a round trip each, 8 us of a
  // 29 us call at n = 8 with the matrices in host memory)
  const cplx* const src = mats + mat0 * (N * N);
  const int nmat = (int)(B - mat0 < MPW ? B - mat0 : MPW), have = nmat * (N * N);
#pragma unroll 1
  for (int e0 = lane; e0 < have; e0 += 64 * 8) {  // lanes of absent matrices walk what LDS holds, and store nothing
    cplx v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = e0 + 64 * u < have ? src[e0 + 64 * u] : cplx{0.0, 0.0};
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int e = e0 + 64 * u, q = e / (N * N), rc = e % (N * N);
      if (e < MPW * N * N) AT[q][(rc % N) * N + rc / N] = v[u];
    }
  }
  __syncthreads();
  const int64_t b = mat0 + gidx;
  const uint32_t start = ((uint32_t)chunk * LPM + (uint32_t)sub) << M;
  if constexpr (perm_is_dd(MODE)) {
    constexpr bool DDCERT = MODE == PERM_DDCERT;
    ddc acc;
    double ea = 0.0;
    auto walk = [&](const cplx* H, const cplx* L, bool exact) __attribute__((always_inline)) {
      if constexpr (DDCERT) {
        glynn_range_ddcert<N>(H, L, start, M, exact, acc, ea);
        cddc_group_sum<LPM>(acc, ea);
      } else {
        glynn_range_dd<N>(H, L, start, M, acc);
        acc = group_sum<LPM>(acc);
      }
    };
    if constexpr (N <= PERM_DD_REG) {
      cplx H[N * N], L[N * N];
      const bool exact = split_own<N>(AT[gidx], H, L);
      walk(H, L, exact);
    } else {
      cplx(&AL)[MPW][N * N] = *reinterpret_cast<cplx(*)[MPW][N * N]>(lds + MPW * N * N);
      __shared__ int inexact[DDCERT ? MPW : 1];
      if constexpr (DDCERT) {
        split_rows<N, MPW, true>(AT, AL, nmat, inexact);
        int bad = inexact[gidx];
        if constexpr (LPM == 64) bad = __builtin_amdgcn_readfirstlane(bad);  // one matrix: in scalar registers
        walk(AT[gidx], AL[gidx], bad == 0);
      } else {
        int none[MPW];
        split_rows<N, MPW, false>(AT, AL, nmat, none);
        walk(AT[gidx], AL[gidx], true);
      }
    }
    if (sub == 0 && b < B) {
      if (W == 1) {
        const double scale = 1.0 / (double)(1ull << (N - 1));
        const ddc sc = ddc_mul_d(acc, scale);  // exact (power of two)
        out[b] = ddc_to_c(sc);
        if constexpr (DDCERT)
          aux[b] = cert_finish(fma(ea, scale, cddc_collapse_err(sc) + 4.0 * CERT_UFL), perm_ddcert_depth(N, M, W));
      } else {
        // chunk partials stay double-double: hi in out, lo in aux-as-cplx,
        // then (certified-dd) the bounds after the B * W lo entries
        out[b * W + chunk] = cplx{acc.re.hi, acc.im.hi};
        reinterpret_cast<cplx*>(aux)[b * W + chunk] = cplx{acc.re.lo, acc.im.lo};
        if constexpr (DDCERT) reinterpret_cast<double*>(reinterpret_cast<cplx*>(aux) + (size_t)B * W)[b * W + chunk] = ea;
      }
    }
  } else {
    constexpr bool KAPPA = (MODE == PERM_KAPPA);
    constexpr bool CERT = (MODE == PERM_CERT);
    cplx acc;
    double aacc;
    glynn_range_fp64<N, C::HOT, KAPPA, CERT>(AT[gidx], start, M, acc, aacc);
    if constexpr (CERT) {
      cert_group_sum<LPM>(acc, aacc);
    } else {
      acc = group_sum<LPM>(acc);
      if (KAPPA) aacc = group_sum<LPM>(aacc);
    }
    if (sub == 0 && b < B) {
      if (W == 1) {
        const double scale = 1.0 / (double)(1ull << (N - 1));
        out[b] = c_scale(acc, scale);
        if (KAPPA) aux[b] = aacc * scale;
        if (CERT) aux[b] = cert_finish(aacc * scale + CERT_UFL, perm_cert_depth(N, M, W));
      } else {
        out[b * W + chunk] = acc;
        if (KAPPA || CERT) aux[b * W + chunk] = aacc;
      }
    }
  }
}

template <int N, int MODE>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(perm_min_waves<MODE>()))) void perm_kernel(
    const cplx* __restrict__ mats, int B, cplx* __restrict__ out, double* __restrict__ aux, int g8, int M, int W) {
  __shared__ cplx lds[perm_lds<N, MODE>()];
  perm_workgroup<N, MODE>(mats, B, out, aux, g8, M, W, blockIdx.x, lds);
}

// Fixed-order (chunk 0, 1, ..., W-1) reduction of chunk partials.
template <int N, int MODE>
__device__ __forceinline__ void perm_reduce(const cplx* __restrict__ part, const double* __restrict__ part_aux, int B,
                                            cplx* __restrict__ out, double* __restrict__ aux, int M, int W,
                                            int64_t b) {
  if (b >= B) return;
  const double scale = 1.0 / (double)(1ull << (N - 1));
  if constexpr (perm_is_dd(MODE)) {
    const cplx* lo = reinterpret_cast<const cplx*>(part_aux);
    const double* pe = reinterpret_cast<const double*>(lo + (size_t)B * W);
    ddc s = ddc_zero();
    double e = 0.0;
    for (int w = 0; w < W; ++w) {
      cplx h = part[b * W + w], l = lo[b * W + w];
      if constexpr (MODE == PERM_DDCERT) {
        double r;
        s = cddc_add(s, ddc{dd{h.re, l.re}, dd{h.im, l.im}}, &r);
        e = e + pe[b * W + w] + r;
      } else {
        s = ddc_add(s, ddc{dd{h.re, l.re}, dd{h.im, l.im}});
      }
    }
    const ddc sc = ddc_mul_d(s, scale);
    out[b] = ddc_to_c(sc);
    if constexpr (MODE == PERM_DDCERT)
      aux[b] = cert_finish(fma(e, scale, cddc_collapse_err(sc) + 4.0 * CERT_UFL), perm_ddcert_depth(N, M, W));
  } else {
    cplx s{0.0, 0.0};
    double a = 0.0;
#pragma unroll 8
    for (int w = 0; w < W; ++w) {  // loads ahead of the serial sum
      s = c_add(s, part[b * W + w]);
      if (MODE == PERM_KAPPA) a += part_aux[b * W + w];
      if (MODE == PERM_CERT) a = cert_round(s, a + part_aux[b * W + w]);
    }
    out[b] = c_scale(s, scale);
    if (MODE == PERM_KAPPA) aux[b] = a * scale;
    if (MODE == PERM_CERT) aux[b] = cert_finish(a * scale + CERT_UFL, perm_cert_depth(N, M, W));
  }
}

template <int N, int MODE>
__global__ void perm_reduce_kernel(const cplx* __restrict__ part, const double* __restrict__ part_aux, int B,
                                   cplx* __restrict__ out, double* __restrict__ aux, int M, int W) {
  perm_reduce<N, MODE>(part, part_aux, B, out, aux, M, W, (int64_t)blockIdx.x * blockDim.x + threadIdx.x);
}

}  // namespace gbsk
