// haf_tree.hpp -- hafnian / loop hafnian of sides N = 14..28 by a subset tree of
// Schur complements over truncated power series (every tier).
//
// The subset sum is the power-trace formula's (haf_impl.hpp): with h = N / 2,
//   haf(A) = sum_S (-1)^(h - |S|) f(S),   f(S) = [eta^h] det(I - eta X A_S)^(-1/2)
//            (loop: times exp(eta/2 d_S^T (X - eta A_S)^-1 d_S), d = diag A),
// X the swap inside each index pair. Where the power-trace form multiplies the
// 2m x 2m matrix of every subset, here subsets share their elimination: in
// M(eta) = X - eta T(eta), T a symmetric matrix of power series (T = A_S at the
// start), eliminating a pair with 2 x 2 block [[a, b], [b, c]] of T leaves
//   T'_jk = T_jk + eta (T_k0 W_j0 + T_k1 W_j1),      W_j = P^-1 (T_j0, T_j1),
//   P^-1 = 1/q [[eta c, u], [u, eta a]], u = 1 - eta b, q = u^2 - eta^2 a c,
// on the remaining rows (the loop vector d is one more row), multiplies the
// determinant by q and adds eta/2 (d_0 W_d0 + d_1 W_d1) to the exponent. The
// logarithmic derivative sigma_k = k [eta^k] log(...) is kept (the power-trace
// formula's kg_k), so the last step is the same Newton recurrence and the terms
// f(S) are the same numbers (kappa keeps its meaning). A tree over include /
// exclude of one pair after another forms each Schur complement once for all
// subsets below it: about 7e6 complex multiply-adds at N = 24 where the
// power-trace form takes 6.5e7. Measured on MI355X, power trace -> tree: N = 16
// (B = 4096) 1099 -> 537 us, N = 24 (B = 256) 3895 -> 1399 us, loop kappa N = 18
// (B = 1001) 1037 -> 488 us, loop dd N = 16 (B = 512) 1789 -> 1350 us; the error
// relative to sum |term| is 0.6-1.0 of the power trace's (loop: 0.3-0.8; dd 0.7-1.0).
// Certified bounds, medians against the power trace's: fp64, complex matrices 0.61 /
// 0.59 / 0.47 / 0.41 / 0.31 / 0.24 at N = 14 .. 24 (loop 0.43 .. 0.17); real ones, where the
// tree's longer sums show, 1.08 / 1.08 / 1.04 at N = 14 / 16 / 18 (single matrices up to
// 3.4), 0.87 and less from 20 on (loop 0.89 and less); dd 1.9 / 2.0 / 1.9 / 1.7 at N = 14 ..
// 20 (loop 1.8 .. 1.1), real 1.8 / 2.3 / 2.5 at N = 14 / 16 / 18 (loop 2.0 / 2.1 / 2.1).
//
// What bounds it: FP64 issue (51-56% of the cycles, 60% of it multiply-adds) and
// the latency between a level's steps, with the waves LDS leaves room for.
//
// The pivot block of every elimination is X + O(eta): its inverse exists as a
// series whatever the entries (no pivoting, no division by data), and every
// step is a sum of products of walk weights, as the matrix powers are.
#pragma once

#include <type_traits>
#include <utility>

#include "cert.hpp"
#include "common.hpp"
#include "haf_parts.hpp"
#include "kernels.hpp"

namespace gbsk {

enum TreeMode { TM_PLAIN = 0, TM_KAPPA = 1, TM_CERT = 2 };

__host__ __device__ constexpr int tree_tri(int r, int c) { return r * (r + 1) / 2 + c; }
// series of a matrix of n pairs: packed lower triangle, then the loop row
__host__ __device__ constexpr int tree_size(bool loop, int n) { return tree_tri(2 * n, 0) + (loop ? 2 * n : 0); }
// first series of level lv's formed matrices (2^(lv-1) of them, T2 - lv pairs each; level 0: the root)
__host__ __device__ constexpr int tree_region(bool loop, int lv) {
  if (lv == 0) return 0;
  int o = tree_size(loop, TREE_T2);
  for (int m = 1; m < lv; ++m) o += (1 << (m - 1)) * tree_size(loop, TREE_T2 - m);
  return o;
}

// Series numbering of one workgroup's LDS: root and formed matrices, then W, then
// q. In fp64 (DD = false) the last level's matrices overwrite W (they are formed
// in registers from it) and, without the loop row, its q stays in registers.
template <bool LOOP, bool DD>
struct TreeSeries {
  static constexpr int ROOT = tree_size(LOOP, TREE_T2);
  static constexpr int W = tree_region(LOOP, TREE_T2 - (DD ? 0 : 1));
  // most W series of a level l: 2^l nodes, 2 (T2 - l - 1) rows (+ the loop row), two components
  static constexpr int NW = LOOP ? 24 : 16;
  static constexpr int Q = W + NW;
  static constexpr int NQ = LOOP || DD ? 8 : 4;
  static constexpr int COUNT = Q + NQ;
  static_assert((1 << (TREE_T2 - 2)) * tree_size(LOOP, 1) <= NW, "the last level's matrices fit W");
  static_assert(COUNT < 256, "series numbers are bytes");
};
constexpr int TREE_SLOTS = 1 << (TREE_T2 - 1);  // sigma slots: the root, then formed matrices (dd: then include leaves)
constexpr int TREE_BX = 15;                     // top coefficients of the in-pair entries: 4, 3, 2 x 2, 4 x 1

// What lane `lane` does at level l: the pivot / row step (two lanes a task: one
// product each in fp64, one component each in dd) and the entry step. Series numbers; TREE_BX for "no top slot".
struct TreeTask {
  uint8_t px, py, w, q;      // product x y, W written, q of the node
  uint8_t sp, sc, b, flags;  // sigma slots of parent and child, top slot of the pivot's b
  uint8_t ew, et, ez, ed;    // entry step: W and T factors, addend, destination
  uint8_t zb, db, esc, pad;  // top slots of addend and destination, sigma slot of E
};
static_assert(sizeof(TreeTask) == 16, "one 16-byte load");
enum { TREE_ON = 1, TREE_PIVOT = 2, TREE_ENTRY = 4, TREE_E = 8 };

template <bool LOOP, bool DD>
struct TreeTable {
  TreeTask t[TREE_T2][64];
  static constexpr int bx_base(int lv) { return lv == 0 ? 0 : (lv == 1 ? 4 : (lv == 2 ? 7 : 11)); }
  constexpr TreeTable() : t{} {
    using S = TreeSeries<LOOP, DD>;
    for (int l = 0; l < TREE_T2; ++l) {
      const bool leaf = l == TREE_T2 - 1;
      const int n = TREE_T2 - l, rows = 2 * (n - 1) + (LOOP ? 1 : 0);
      // node v of level l reads the matrix its last include formed (level lv,
      // number g there), two rows further down per exclude since
      struct Node {
        int base = 0, sh = 0, slot = 0, bx = 0;
      };
      auto node = [&](int v) constexpr {
        Node r;
        if (v == 0) {
          r.sh = 2 * l;
          r.bx = l;
          return r;
        }
        int p = 0;
        while (!((v >> p) & 1)) ++p;
        const int lv = l - p, g = v >> (p + 1);
        r.base = tree_region(LOOP, lv) + g * tree_size(LOOP, TREE_T2 - lv);
        r.sh = 2 * p;
        r.slot = (1 << (lv - 1)) + g;
        r.bx = bx_base(lv) + g * (TREE_T2 - lv) + p;
        return r;
      };
      auto at = [&](const Node& r, int i, int j) constexpr { return r.base + tree_tri(i + r.sh, j + r.sh); };
      for (int lane = 0; lane < 64; ++lane) {
        TreeTask& k = t[l][lane];
        const int half = lane & 1, pl = lane >> 1, tpn = 1 + 2 * rows;
        k.b = k.zb = k.db = TREE_BX;
        if (pl < (tpn << l)) {
          const int nu = pl / tpn, task = pl % tpn;
          const Node r = node(nu);
          const int a = at(r, 0, 0), b = at(r, 1, 0), c = at(r, 1, 1);
          k.flags = TREE_ON;
          if (task == 0) {
            k.flags |= TREE_PIVOT;
            k.px = half ? a : b;
            k.py = half ? c : b;
            k.b = r.bx;
          } else {
            const int j = 2 + (task - 1) / 2, c0 = (task - 1) % 2 == 0;
            const int x = at(r, j, 0), y = at(r, j, 1);
            k.px = half ? b : (c0 ? c : a);
            k.py = half == c0 ? y : x;
            k.w = S::W + nu * rows * 2 + task - 1;
          }
          k.q = S::Q + nu;
          k.sp = r.slot;
          k.sc = (1 << l) + nu;
        }
        const int r0 = 2 * (n - 1), ne = tree_size(LOOP, n - 1), epn = ne + (LOOP ? 1 : 0);
        if ((!leaf || (LOOP && DD)) && pl < (epn << l)) {
          const int nv = pl / epn, e = pl % epn;
          const Node r = node(nv);
          int i = 0;
          while (tree_tri(i + 1, 0) <= e && i < r0) ++i;
          int j = e - tree_tri(i, 0);
          k.flags |= TREE_ENTRY;
          if (LOOP && e == ne) {
            k.flags |= TREE_E;
            i = j = r0;
          }
          k.ew = S::W + (nv * rows + i) * 2 + half;
          k.et = at(r, j + 2, half);
          k.ez = (k.flags & TREE_E) ? 0 : at(r, i + 2, j + 2);
          k.ed = tree_region(LOOP, l + 1) + nv * ne + ((k.flags & TREE_E) ? 0 : e);
          k.esc = (1 << l) + nv;
          if (i < r0 && (i & 1) && j == i - 1) {
            k.zb = r.bx + 1 + i / 2;
            k.db = bx_base(l + 1) + nv * (n - 1) + i / 2;
          }
        }
      }
    }
  }
};
template <bool LOOP, bool DD>
__device__ constexpr TreeTable<LOOP, DD> tree_table{};

// ------------------------------------------------------------ lane exchanges
// lane U of each row of 16 lanes to the whole row (one 64-bit DPP move)
template <int U>
__device__ __forceinline__ double row_bcast_d(double v) {
  return __builtin_bit_cast(
      double, (long long)__builtin_amdgcn_update_dpp(0ll, __builtin_bit_cast(long long, v), 0x150 + U, 0xF, 0xF, true));
}
template <int U>
__device__ __forceinline__ cplx row_bcast(cplx v) {
  return cplx{row_bcast_d<U>(v.re), row_bcast_d<U>(v.im)};
}
__device__ __forceinline__ cplx swap_pair_c(cplx a) { return cplx{swap_pair_d(a.re), swap_pair_d(a.im)}; }
// the values of lanes 0..31 and of lanes 32..63, each in both halves of the wave
__device__ __forceinline__ void halves_d(double v, double& lo, double& hi) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned x = (unsigned)b, y = (unsigned)(b >> 32);
  const auto rx = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  const auto ry = __builtin_amdgcn_permlane32_swap(y, y, false, false);
  lo = __builtin_bit_cast(double, ((unsigned long long)ry[0] << 32) | rx[0]);
  hi = __builtin_bit_cast(double, ((unsigned long long)ry[1] << 32) | rx[1]);
}

// LDS layout of one workgroup in complex (dd: complex double-double) numbers. Stored series have KC
// coefficients, KS (odd: bank spread) slots apart: degrees 0 .. H - 2 (the top
// degree H - 1 only of the in-pair entries b, in BX), with the loop row 0 .. H - 1.
template <bool LOOP, int H, bool DD>
struct TreeLds {
  using S = TreeSeries<LOOP, DD>;
  static constexpr int KC = LOOP ? H : H - 1;
  static constexpr int KS = KC | 1;
  static constexpr int S0 = S::COUNT * KS;              // sigma, H coefficients a slot
  static constexpr int B0 = S0 + (DD ? 2 : 1) * TREE_SLOTS * H;        // top coefficients (not with the loop row)
  static constexpr int TOTAL = B0 + (LOOP ? 0 : TREE_BX + 1);
  // leading-pair elimination, after the root: V columns (two buffers), trace shares, E
  static constexpr int PM = 2 * (H - TREE_T2);
  static constexpr int RR = 2 * TREE_T2 + (LOOP ? 1 : 0);
  static constexpr int V0 = S::ROOT * KS, VN = PM * RR;
  static constexpr int PB0 = V0 + 2 * VN;
  static constexpr int E0 = PB0 + (H + 1) * PM;
  static_assert(E0 + (LOOP ? H + 1 : 0) <= S0, "the leading-pair scratch ends before the root's sigma");
  static_assert(PM + RR <= 32, "one column a lane of each half wave");
};

// Certified bounds (of the modulus; model and bound arithmetic: cert.hpp): every
// value formed here is a chain acc = c_fma(x_i, y_i, acc) plus single operations on
// its result. One step's four roundings (common.hpp c_fma: the products with Im x
// go first) are at most
//   u (|acc_before| + |Im x_i| |y_i|) + u |acc_after|   (up to the factor 1 + u);
// so a step charges 2 u |acc_before| and
//   |x| ey + ex (|y| + ey) + u |Im x| |y| = (|x| + ex) ey + (ex + u |Im x|) |y|
// for its operands' bounds ex, ey, the chain's end u |acc|, and each further
// operation its own rounding u |result|. TREE_U carries the factors 1 + u,
// TREE_UFL the underflows of a chain. Roundings take |Re| + |Im| for |z|; the factors
// of a bound take tree_abs, since products nest deeper here than in the power trace
// and |Re| + |Im| is 1.27 |z| on average: with it bounds were 3 times as wide.
constexpr double TREE_UFL = 1e-317;
constexpr double TREE_U = CERT_U * 1.0000001;
// |a + ib| from above: the chord of sqrt(1 + t^2) over t = 0 .. 1, at most 8% more. A NaN may
// be dropped: it is in the value as well, whose own rounding then refuses the bound.
__host__ __device__ __forceinline__ double tree_abs(double a, double b) {
  return fma(0.41421356237309515, fmin(fabs(a), fabs(b)), fmax(fabs(a), fabs(b)));
}
__host__ __device__ __forceinline__ double tree_abs(cplx z) { return tree_abs(z.re, z.im); }
__host__ __device__ __forceinline__ double tree_rnd(cplx z, double e) { return fma(TREE_U, cert_norm1(z), e); }
__host__ __device__ __forceinline__ double tree_im(cplx x, double ex) { return fma(TREE_U, fabs(x.im), ex); }
// one certified chain step: xs = |x| + ex, xr = ex + u |Im x| of the x operand, Y = |y|
template <bool CERT>
__host__ __device__ __forceinline__ void tree_mac(cplx& acc, double& e, const cplx& x, double xs, double xr, const cplx& y,
                                         double ey, double Y) {
  if constexpr (CERT) e = fma(2.0 * TREE_U, cert_norm1(acc), fma(xs, ey, fma(xr, Y, e)));
  acc = c_fma(x, y, acc);
}
// acc = x y, coefficients 0 .. H - 1, one chain each: x(i, value, bound) reads x
template <bool CERT, int H, class X>
__host__ __device__ __forceinline__ void tree_product(const X& x, const cplx (&y)[H], const double (&ey)[CERT ? H : 1],
                                                      cplx (&acc)[H], double (&ea)[CERT ? H : 1]) {
  double Y[CERT ? H : 1];
#pragma unroll
  for (int d = 0; d < H; ++d) {
    acc[d] = cplx{0.0, 0.0};
    if constexpr (CERT) {
      Y[d] = tree_abs(y[d]);
      ea[d] = TREE_UFL;
    }
  }
#pragma unroll
  for (int i = 0; i < H; ++i) {
    cplx a;
    double e = 0.0;
    x(i, a, e);
    const double xs = tree_abs(a) + e, xr = tree_im(a, e);
#pragma unroll
    for (int d = i; d < H; ++d)
      tree_mac<CERT>(acc[d], ea[CERT ? d : 0], a, xs, xr, y[d - i], ey[CERT ? d - i : 0], Y[CERT ? d - i : 0]);
  }
  if constexpr (CERT) {
#pragma unroll
    for (int d = 0; d < H; ++d) ea[d] = tree_rnd(acc[d], ea[d]);
  }
}
// the bound arithmetic itself is at most this many roundings deep (cert_finish):
// four levels of three chains, each a recurrence of depth at most 4 H^2, and
// the leading pairs' H / 2 products
constexpr double TREE_DEPTH = 65536.0;

// s += sum over the included pairs' columns u of C[row][u] x[u]: the row of C lies
// across each 16 lanes (columns 16 .. in c2); es += |C| ex in the certified mode
template <int PM, bool CERT, int... Ps>
__device__ __forceinline__ void tree_row(cplx& s, double& es, const cplx& c, const cplx& c2, const cplx (&x)[PM],
                                         const double (&ex)[CERT ? PM : 1], int k1, std::integer_sequence<int, Ps...>) {
  auto term = [&](const cplx& z, int u) __attribute__((always_inline)) {
    if constexpr (CERT) es = fma(2.0 * TREE_U, cert_norm1(s), fma(tree_abs(z), ex[u], es));
    s = c_fma(z, x[u], s);
  };
  (((Ps < k1) ? (term(row_bcast<(2 * Ps) % 16>(Ps < 8 ? c : c2), 2 * Ps),
                 term(row_bcast<(2 * Ps + 1) % 16>(Ps < 8 ? c : c2), 2 * Ps + 1), 0)
              : 0),
   ...);
}

// True in every lane if an entry the value depends on is not finite. The
// elimination reads the leading rows and one triangle of the trailing block; the
// workgroup without leading pairs, which has the least to do, looks at the rest,
// so an entry of either triangle makes the value NaN.
template <bool LOOP, int N>
__device__ __forceinline__ bool tree_nonfinite(const cplx* __restrict__ A) {
  bool bad = false;
  for (int e = threadIdx.x; e < N * N; e += 64) {
    const cplx z = A[e];
    if (LOOP || e % (N + 1) != 0) bad |= !(fabs(z.re) < INFINITY && fabs(z.im) < INFINITY);
  }
  return __any(bad);
}

// One workgroup: instance b, include pattern p1 of the H - T2 leading pairs.
template <bool LOOP, int H, int MODE>
__global__ __launch_bounds__(64) void haf_tree_kernel(const cplx* __restrict__ mats, cplx* __restrict__ part,
                                                      double* __restrict__ part_abs) {
  using L = TreeLds<LOOP, H, false>;
  using S = TreeSeries<LOOP, false>;
  constexpr int T2 = TREE_T2, KC = L::KC, KS = L::KS, N = 2 * H, T1 = H - T2, RR = L::RR, PM = L::PM;
  constexpr bool KAPPA = MODE == TM_KAPPA, CERT = MODE == TM_CERT;
  __shared__ cplx lds[L::TOTAL];
  __shared__ double ldse[CERT ? L::TOTAL : 1];  // bounds, at the same places
  const int lane = threadIdx.x;
  const int64_t b = (int64_t)blockIdx.x >> T1;
  const unsigned p1 = blockIdx.x & ((1u << T1) - 1u);
  const int k1 = __popc(p1);
  const cplx* __restrict__ A = mats + b * N * N;
  cplx* const sig = lds + L::S0;
  double* const sige = ldse + (CERT ? L::S0 : 0);
  cplx* const bx = lds + (LOOP ? 0 : L::B0);
  double* const bxe = ldse + (CERT && !LOOP ? L::B0 : 0);
  TreeTask task[T2];
#pragma unroll
  for (int l = 0; l < T2; ++l) task[l] = tree_table<LOOP, false>.t[l][lane];

  // ---- leading pairs: with C = X T_pp and V_j = C^j X T_pr (columns: the
  // trailing rows, then the loop vector), T' = T_rr + sum_i eta^(i+1) V_a^T X V_b,
  // a + b = i, since (C^a X T_pr)^T = T_rp C^a X; tr(C^k) / 2 and k/2 V_d^T X V_d
  // are the root's sigma. Rows 2i, 2i + 1 belong to the i-th included pair. A lane
  // holds one column of (C^(j+1) | V_j) in registers, the same in both halves of
  // the wave; half 0 forms the even rows of the next one, half 1 the odd rows,
  // C's entries coming from the lanes of each row of 16 by DPP.
  int ei = 0, ej = 0;  // this lane's root entry
  {
    while (tree_tri(ei + 1, 0) <= lane && ei < 2 * T2) ++ei;
    ej = lane - tree_tri(ei, 0);
  }
  const bool mine = lane < S::ROOT, top = !LOOP && mine && (ei & 1) && ej == ei - 1;
  // coefficient k of the root entry: the stored series, or the top slot
  auto put = [&](int k, cplx v, double e) __attribute__((always_inline)) {
    if (k < KC) {
      lds[lane * KS + k] = v;
      if constexpr (CERT) ldse[lane * KS + k] = e;
    } else if (k < H && top) {
      bx[ei >> 1] = v;
      if constexpr (CERT) bxe[ei >> 1] = e;
    }
  };
  if (mine) {
    const int r = PM + ej, i = ei < 2 * T2 ? PM + ei : r;
    put(0, (!LOOP && i == r) ? cplx{0.0, 0.0} : A[i * N + r], 0.0);
  }
  const bool off = p1 == 0 && tree_nonfinite<LOOP, N>(A);
  if (p1 == 0) {
    if (mine) {
      for (int k = 1; k < H; ++k) put(k, cplx{0.0, 0.0}, 0.0);
    }
    if (lane < H) {
      sig[lane] = cplx{0.0, 0.0};
      if constexpr (CERT) sige[lane] = 0.0;
    }
  } else {
    cplx cur[PM], nxt[PM];
    double ecur[CERT ? PM : 1], enxt[CERT ? PM : 1];  // bounds
    cplx cr[T1], cr2[PM > 16 ? T1 : 1];  // this half's row of C of each pair: columns lane % 16, 16 + lane % 16
    const int hf = lane >> 5, col = lane & 31;
    const int vcol = col - (32 - RR);  // V columns: the last RR lanes of a half
    const bool isv = vcol >= 0, isc = col < 2 * k1;
    int pr[T1];                   // leading pairs included, in order
    int ac = 0, au = 0, au2 = 0;  // rows of A of columns col, lane % 16, 16 + lane % 16
    {
      unsigned rest = p1;
#pragma unroll
      for (int i = 0; i < T1; ++i) {
        pr[i] = rest ? 2 * __builtin_ctz(rest) : 0;
        rest &= rest - 1;
        if ((col >> 1) == i) ac = pr[i] + (col & 1);
        if (((lane & 15) >> 1) == i) au = pr[i] + (lane & 1);
        if (PM > 16 && 8 + ((lane & 15) >> 1) == i) au2 = pr[i] + (lane & 1);
      }
    }
    if (isv) ac = PM + vcol;
    int vc = L::V0, vn = L::V0 + L::VN;
#pragma unroll
    for (int t = 0; t < PM; ++t) {
      nxt[t] = cur[t] = cplx{0.0, 0.0};
      if constexpr (CERT) enxt[t] = ecur[t] = 0.0;
      if ((t >> 1) < k1) {
        const int r = pr[t >> 1] + ((t & 1) ^ 1);
        const cplx a = A[r * N + ((LOOP && vcol == 2 * T2) ? r : ac)];
        if ((isc || isv) && (LOOP || ac != r)) cur[t] = a;
      }
    }
#pragma unroll
    for (int i = 0; i < T1; ++i) {
      if (i < k1) {
        const int r = pr[i] + 1 - hf;
        cr[i] = (!LOOP && au == r) ? cplx{0.0, 0.0} : A[r * N + au];
        if constexpr (PM > 16) cr2[i] = (!LOOP && au2 == r) ? cplx{0.0, 0.0} : A[r * N + au2];
      }
    }
    if (isv && hf == 0) {
#pragma unroll
      for (int t = 0; t < PM; ++t)
        if ((t >> 1) < k1) {
          lds[vc + t * RR + vcol] = cur[t];
          if constexpr (CERT) ldse[vc + t * RR + vcol] = 0.0;
        }
    }
    constexpr int J = (H + 1) / 2;
#pragma unroll 1
    for (int j = 0; j < J; ++j) {
      {
        double yA[CERT ? PM : 1];  // C is exact: |C| (e + u |x|)
        if constexpr (CERT) {
#pragma unroll
          for (int t = 0; t < PM; ++t) yA[t] = tree_rnd(cur[t], ecur[t]);
        }
#pragma unroll
        for (int i = 0; i < T1; ++i)
          if (i < k1) {
            cplx s{0.0, 0.0};
            double es = TREE_UFL;
            tree_row<PM, CERT>(s, es, cr[i], cr2[PM > 16 ? i : 0], cur, yA, k1, std::make_integer_sequence<int, T1>{});
            halves_d(s.re, nxt[2 * i].re, nxt[2 * i + 1].re);
            halves_d(s.im, nxt[2 * i].im, nxt[2 * i + 1].im);
            if constexpr (CERT) halves_d(tree_rnd(s, es), enxt[2 * i], enxt[2 * i + 1]);
          }
      }
      if (isv && hf == 0) {
#pragma unroll
        for (int t = 0; t < PM; ++t)
          if ((t >> 1) < k1) {
            lds[vn + t * RR + vcol] = nxt[t];
            if constexpr (CERT) ldse[vn + t * RR + vcol] = enxt[t];
          }
      }
      // tr(C^a C^b) = sum C^a[t][c] C^b[t^1][c^1] (rows 2i and 2i + 1 give the same when a = b)
      cplx pe{0.0, 0.0}, po{0.0, 0.0};
      double epe = TREE_UFL, epo = TREE_UFL;
      auto term = [&](cplx& s, double& es, const cplx& x, double ex, const cplx& y, double ey)
                      __attribute__((always_inline)) {
        tree_mac<CERT>(s, es, x, tree_abs(x) + ex, tree_im(x, ex), y, ey, tree_abs(y));
      };
#pragma unroll
      for (int i = 0; i < T1; ++i)
        if (i < k1) {
          const int t = 2 * i;
          const cplx y = swap_pair_c(cur[t + 1]), z = swap_pair_c(nxt[t + 1]);
          const double ey = CERT ? swap_pair_d(ecur[CERT ? t + 1 : 0]) : 0.0;
          const double ez = CERT ? swap_pair_d(enxt[CERT ? t + 1 : 0]) : 0.0;
          const double ex = CERT ? ecur[CERT ? t : 0] : 0.0, en = CERT ? enxt[CERT ? t : 0] : 0.0;
          term(pe, epe, cur[t], ex, y, ey);
          term(po, epo, cur[t], ex, z, ez);
          term(po, epo, nxt[t], en, y, ey);
        }
      if (isc && hf == 0) {
        const int o = L::PB0 + (2 * j + 1) * PM + col;
        lds[o] = c_scale(pe, 2.0);  // tr C^(2j+2)
        if constexpr (CERT) ldse[o] = 2.0 * tree_rnd(pe, epe);
        if (2 * j + 2 < H) {
          lds[o + PM] = po;
          if constexpr (CERT) ldse[o + PM] = tree_rnd(po, epo);
        }
      }
      __syncthreads();
      if (mine || (LOOP && lane == S::ROOT)) {
        cplx s1{0.0, 0.0}, s2{0.0, 0.0};
        double e1 = TREE_UFL, e2 = TREE_UFL;
#pragma unroll 2
        for (int i = 0; i < k1; ++i) {
          const int o = 2 * i * RR;
          auto at = [&](int q, cplx& z, double& e) __attribute__((always_inline)) {
            z = lds[q];
            e = CERT ? ldse[CERT ? q : 0] : 0.0;
          };
          cplx x0, x1, y0, y1, z0, z1;
          double f0, f1, g0, g1, h0, h1;
          at(vc + o + ei, x0, f0);
          at(vc + o + RR + ei, x1, f1);
          at(vc + o + ej, y0, g0);
          at(vc + o + RR + ej, y1, g1);
          at(vn + o + ej, z0, h0);
          at(vn + o + RR + ej, z1, h1);
          term(s1, e1, x0, f0, y1, g1);
          term(s1, e1, x1, f1, y0, g0);
          term(s2, e2, x0, f0, z1, h1);
          term(s2, e2, x1, f1, z0, h0);
        }
        e1 = tree_rnd(s1, e1);
        e2 = tree_rnd(s2, e2);
        if (LOOP && lane == S::ROOT) {
          lds[L::E0 + 2 * j] = s1;
          lds[L::E0 + 2 * j + 1] = s2;
          if constexpr (CERT) {
            ldse[L::E0 + 2 * j] = e1;
            ldse[L::E0 + 2 * j + 1] = e2;
          }
        } else {
          put(2 * j + 1, s1, e1);
          put(2 * j + 2, s2, e2);
        }
      }
      __syncthreads();
#pragma unroll
      for (int t = 0; t < PM; ++t) {
        cur[t] = nxt[t];
        if constexpr (CERT) ecur[t] = enxt[t];
      }
      const int sw = vc;
      vc = vn;
      vn = sw;
    }
    if (lane < H) {
      cplx s{0.0, 0.0};
      double e = TREE_UFL;
      auto add = [&](const cplx& x, double ex) __attribute__((always_inline)) {
        s = c_add(s, x);
        if constexpr (CERT) e = cert_round(s, e + ex);
      };
      if (lane == 0) {
        for (unsigned rest = p1; rest; rest &= rest - 1) {  // tr C
          const int t = 2 * __builtin_ctz(rest);
          add(A[t * N + t + 1], 0.0);
          add(A[(t + 1) * N + t], 0.0);
        }
      } else {
        for (int i = 0; i < 2 * k1; ++i) {
          const int o = L::PB0 + lane * PM + i;
          add(lds[o], CERT ? ldse[CERT ? o : 0] : 0.0);
        }
      }
      s = c_scale(s, 0.5);
      e = fma(0.5, e, TREE_UFL);
      if constexpr (LOOP) {
        const cplx v = c_scale(lds[L::E0 + lane], 0.5 * (lane + 1));
        add(v, CERT ? cert_round(v, 0.5 * (lane + 1) * ldse[CERT ? L::E0 + lane : 0]) : 0.0);
      }
      sig[lane] = s;
      if constexpr (CERT) sige[lane] = e;
    }
  }
  __syncthreads();

  // ---- the tree: level l has 2^l nodes of T2 - l pairs; tree_table says what each
  // lane does. Only include children are formed: an exclude child is its parent
  // read two rows further down (the packed index does not depend on the size).
  // A task's two products go to lanes 2i, 2i + 1.
  const int half = lane & 1;
  cplx coeff{0.0, 0.0};
  double ecoeff = 0.0;
  bool live = false;
#pragma unroll
  for (int l = 0; l < T2; ++l) {
    const bool leaf = l == T2 - 1;
    const TreeTask k = task[l];
    const bool on = k.flags & TREE_ON, isq = k.flags & TREE_PIVOT;
    // v = m P + eta (x1 y1 - x2 y2): rows c x - b y, a y - b x over P = y, x; the
    // pivot task b b - a c over P = b, m = -2 gives q_1, q_2, ...; the addend
    // m P is one of the two lanes' y operand
    cplx v[H], y[H];
    double ev[CERT ? H : 1], yA[CERT ? H : 1], yB[CERT ? H : 1];
    // v[d + sh] += sum x_i y_(d - i), d < n, over the x at series px (sign sg)
    if (on) {
      const cplx* const px = lds + k.px * KS;
      const cplx* const py = lds + k.py * KS;
      const double m = isq ? (half ? 0.0 : -2.0) : (half ? 1.0 : 0.0);
      const double sg = half ? -1.0 : 1.0;
#pragma unroll
      for (int d = 0; d < H; ++d) {
        y[d] = d < KC ? py[d] : bx[k.b];
        v[d] = cplx{0.0, 0.0};
        if constexpr (CERT) {
          const double ey = d < KC ? ldse[k.py * KS + d] : bxe[k.b], Y = tree_abs(y[d]);
          yA[d] = ey;
          yB[d] = Y;
          ev[d] = fma(fabs(m), ey, TREE_UFL);
        }
      }
#pragma unroll
      for (int i = 0; i < H - 1; ++i) {
        const cplx x = c_scale(px[i], sg);
        const double ex = CERT ? ldse[CERT ? k.px * KS + i : 0] : 0.0;
        const double xs = tree_abs(x) + ex, xr = tree_im(x, ex);
#pragma unroll
        for (int d = i; d < H - 1; ++d)
          tree_mac<CERT>(v[d + 1], ev[CERT ? d + 1 : 0], x, xs, xr, y[d - i], yA[CERT ? d - i : 0], yB[CERT ? d - i : 0]);
      }
#pragma unroll
      for (int d = 0; d < H; ++d) {
        if constexpr (CERT) ev[d] = tree_rnd(v[d], ev[d]);
        v[d] = c_axpy(m, y[d], v[d]);
        if constexpr (CERT) ev[d] = tree_rnd(v[d], ev[d]);
        v[d] = c_add(v[d], swap_pair_c(v[d]));
        if constexpr (CERT) ev[d] = tree_rnd(v[d], ev[d] + swap_pair_d(ev[d]));
      }
    }
    const bool shareq = !leaf || LOOP;  // row tasks read their node's q
    if (shareq) {
      if (on && isq && !half) {
#pragma unroll
        for (int d = 0; d < KC; ++d) {
          lds[k.q * KS + d] = v[d];
          if constexpr (CERT) ldse[k.q * KS + d] = ev[d];
        }
      }
      __syncthreads();
    }
    // q y = v: W of the row tasks; the pivot task's right-hand side
    // -eta q' / 2 gives its share of sigma (sigma_(k+1) at index k)
    if (on) {
#pragma unroll
      for (int d = 0; d < H - 1; ++d) {
        y[d] = c_neg(shareq ? lds[k.q * KS + d] : v[d]);
        if constexpr (CERT) {
          const double ey = shareq ? ldse[k.q * KS + d] : ev[d], Y = tree_abs(y[d]);
          yA[d] = ey;
          yB[d] = Y;
        }
      }
#pragma unroll
      for (int d = 0; d < H; ++d) {
        const double s = isq ? -0.5 * (d + 1) : 1.0;
        v[d] = c_scale(v[d], s);
        if constexpr (CERT) ev[d] = isq ? tree_rnd(v[d], fabs(s) * ev[d]) : ev[d];
      }
#pragma unroll
      for (int i = 1; i < H; ++i) {
        const cplx x = v[i - 1];
        // v[0] is no chain
        if constexpr (CERT) ev[i - 1] = i > 1 ? tree_rnd(x, ev[i - 1]) : ev[0];
        const double ex = CERT ? ev[CERT ? i - 1 : 0] : 0.0;
        const double xs = tree_abs(x) + ex, xr = tree_im(x, ex);
#pragma unroll
        for (int d = i; d < H; ++d)
          tree_mac<CERT>(v[d], ev[CERT ? d : 0], x, xs, xr, y[d - i], yA[CERT ? d - i : 0], yB[CERT ? d - i : 0]);
      }
      if constexpr (CERT) ev[H - 1] = tree_rnd(v[H - 1], ev[H - 1]);
      if (!isq && !half && !leaf) {
#pragma unroll
        for (int d = 0; d < KC; ++d) {
          lds[k.w * KS + d] = v[d];
          if constexpr (CERT) ldse[k.w * KS + d] = ev[d];
        }
      }
      if (isq) {  // the child's sigma; at the last level the include leaf's (even lane), the odd lane takes the exclude leaf
#pragma unroll
        for (int d = 0; d < H; ++d) {
          const cplx p = sig[k.sp * H + d];
          const cplx s = c_add(p, v[d]);
          const double es = CERT ? cert_round(s, sige[CERT ? k.sp * H + d : 0] + ev[CERT ? d : 0]) : 0.0;
          if (leaf) {
            v[d] = half ? p : s;
            if constexpr (CERT) ev[d] = half ? sige[k.sp * H + d] : es;
          } else if (!half) {
            sig[k.sc * H + d] = s;
            if constexpr (CERT) sige[k.sc * H + d] = es;
          }
        }
      }
    }
    if (!leaf) {
      __syncthreads();
      // form the include children: entry (i, j) = T_ij + eta (T_j0 W_i0 + T_j1 W_i1);
      // with the loop row also E = d_0 W_d0 + d_1 W_d1, a share of the child's sigma
      const bool eon = k.flags & TREE_ENTRY, isE = k.flags & TREE_E;
      cplx acc[KC], z[H];
      double ea[CERT ? KC : 1], ez[CERT ? H : 1];
      if (eon) {
#pragma unroll
        for (int d = 0; d < KC; ++d) {
          y[d] = lds[k.ew * KS + d];
          acc[d] = cplx{0.0, 0.0};
          if constexpr (CERT) {
            const double ey = ldse[k.ew * KS + d], Y = tree_abs(y[d]);
            yA[d] = ey;
            yB[d] = Y;
            ea[d] = TREE_UFL;
          }
        }
#pragma unroll
        for (int i = 0; i < KC; ++i) {
          const cplx x = lds[k.et * KS + i];
          const double ex = CERT ? ldse[CERT ? k.et * KS + i : 0] : 0.0;
          const double xs = tree_abs(x) + ex, xr = tree_im(x, ex);
#pragma unroll
          for (int d = i; d < KC; ++d)
            tree_mac<CERT>(acc[d], ea[CERT ? d : 0], x, xs, xr, y[d - i], yA[CERT ? d - i : 0], yB[CERT ? d - i : 0]);
        }
#pragma unroll
        for (int d = 0; d < KC; ++d) {
          if constexpr (CERT) ea[d] = tree_rnd(acc[d], ea[d]);
          acc[d] = c_add(acc[d], swap_pair_c(acc[d]));
          if constexpr (CERT) ea[d] = tree_rnd(acc[d], ea[d] + swap_pair_d(ea[d]));
        }
        if (!half && !isE) {
#pragma unroll
          for (int d = 0; d < H; ++d) {
            z[d] = d < KC ? lds[k.ez * KS + d] : bx[k.zb];
            if constexpr (CERT) ez[d] = d < KC ? ldse[k.ez * KS + d] : bxe[k.zb];
          }
        }
      }
      if (l == T2 - 2) __syncthreads();  // the last level's matrices overwrite W
      if (eon && !half) {
        if (isE) {
#pragma unroll
          for (int d = 0; d < KC; ++d) {
            const double s = 0.5 * (d + 1);
            const cplx x = c_scale(acc[d], s);
            const int o = k.esc * H + d;
            const cplx t = c_add(sig[o], x);
            sig[o] = t;
            if constexpr (CERT) sige[o] = cert_round(t, sige[o] + fma(s, ea[d], 2.0 * CERT_U * cert_norm1(x)));
          }
        } else {
#pragma unroll
          for (int d = 0; d < H; ++d) {
            const cplx t = d ? c_add(z[d], acc[d ? d - 1 : 0]) : z[0];
            const double et = CERT ? (d ? tree_rnd(t, ez[CERT ? d : 0] + ea[CERT && d ? d - 1 : 0]) : ez[0]) : 0.0;
            if (d < KC) {
              lds[k.ed * KS + d] = t;
              if constexpr (CERT) ldse[k.ed * KS + d] = et;
            } else {
              bx[k.db] = t;  // TREE_BX: a slot nothing reads
              if constexpr (CERT) bxe[k.db] = et;
            }
          }
        }
      }
      __syncthreads();
    } else {
      if constexpr (LOOP) {
        // E of the include leaves: the loop row's task lanes multiply their W (in
        // registers) with d_0 or d_1 (half 0's y operand) and hand it over through W
        cplx acc[H];
        double ea[CERT ? H : 1];
        if (on && !isq)
          tree_product<CERT, H>(
              [&](int i, cplx& x, double& ex) __attribute__((always_inline)) {
                x = lds[k.py * KS + i];
                if constexpr (CERT) ex = ldse[k.py * KS + i];
              },
              v, ev, acc, ea);
        __syncthreads();
        if (on && !isq && !half) {
#pragma unroll
          for (int d = 0; d < H; ++d) {
            lds[k.w * KS + d] = acc[d];
            if constexpr (CERT) ldse[k.w * KS + d] = ea[d];
          }
        }
        __syncthreads();
        if (on && isq && !half) {
          const int w = S::W + 2 * (k.q - S::Q);
#pragma unroll
          for (int d = 0; d < H; ++d) {
            const double s = 0.5 * (d + 1);
            const cplx x = c_scale(c_add(lds[w * KS + d], lds[(w + 1) * KS + d]), s);
            v[d] = c_add(v[d], x);
            if constexpr (CERT)
              ev[d] = cert_round(v[d], ev[d] + fma(s, ldse[w * KS + d] + ldse[(w + 1) * KS + d], 4.0 * CERT_U * cert_norm1(x)));
          }
        }
      }
      // Newton: e_j = (1/j) sum_k sigma_k e_(j-k), the odd lane on the exclude leaf
      live = on && isq;
      if (live) {
        cplx s[H + 1];
        double es[CERT ? H + 1 : 1];
#pragma unroll
        for (int j = 0; j <= H; ++j) {
          s[j] = cplx{0.0, 0.0};
          if constexpr (CERT) es[j] = TREE_UFL;
        }
        if constexpr (CERT) {
#pragma unroll
          for (int d = 0; d < H; ++d) {
            const double Y = tree_abs(v[d]);
            yA[d] = ev[d];
            yB[d] = Y;
          }
        }
#pragma unroll
        for (int j = 0; j <= H; ++j) {
          cplx e{1.0, 0.0};
          double ee = 0.0;
          if (j) {
            // s / j: the rounded reciprocal's quotient, corrected by its residual
            const double r = 1.0 / j;
            e = c_scale(s[j], r);
            e.re = fma(fma(-(double)j, e.re, s[j].re), r, e.re);
            e.im = fma(fma(-(double)j, e.im, s[j].im), r, e.im);
            if constexpr (CERT) ee = fma(tree_rnd(s[j], es[j]), (1.0 + 8.0 * CERT_U) / j, 4.0 * CERT_U * cert_norm1(e));
          }
          const double xs = tree_abs(e) + ee, xr = tree_im(e, ee);
          if (j == H) {
            coeff = e;
            ecoeff = ee;
          }
#pragma unroll
          for (int t = j + 1; t <= H; ++t)
            tree_mac<CERT>(s[t], es[CERT ? t : 0], e, xs, xr, v[t - j - 1], yA[CERT ? t - j - 1 : 0],
                           yB[CERT ? t - j - 1 : 0]);
        }
        const int nsel = k1 + __popc((unsigned)(k.q - S::Q)) + (half ? 0 : 1);
        if ((H - nsel) & 1) coeff = c_neg(coeff);
      }
    }
  }
  if (!live) {
    coeff = cplx{0.0, 0.0};
    ecoeff = 0.0;
  }
  double a = 0.0;
  if constexpr (KAPPA) a = group_sum<64>(c_abs(coeff));
  if constexpr (CERT) {
    cert_group_sum<64>(coeff, ecoeff);
    a = cert_finish(ecoeff, TREE_DEPTH);
  } else {
    coeff = group_sum<64>(coeff);
  }
  if (lane == 0) {
    part[blockIdx.x] = off ? cplx{NAN, NAN} : coeff;
    if constexpr (KAPPA || CERT) part_abs[blockIdx.x] = off ? (CERT ? INFINITY : NAN) : a;
  }
}

// ------------------------------------------------------------- double-double
// The same tree with complex double-double series; a task's two lanes form the
// real and the imaginary part of all its coefficients. A chain of real products
// starts from the value it adds to and keeps three words: high and low words are
// summed by TwoSum, the low words' errors in lo2 (18 operations a product; 19 take a
// normalised product and a sum), so a product leaves three roundings at the
// 2^-106 level, those of its cross terms and of t. With the low words summed in
// one double (12 operations, 0.85 of the time) results were 1.2-1.8 times as far
// from quad values as the power trace's; this is 0.55-0.96 of it (N = 14 .. 20).
// R: r receives the chain's own error: those roundings and the product of the low
// words, which is not formed, and at the end the rounding of w and, where |w| >
// |h.hi|, the last FastTwoSum's (a = h.hi, b = w: fl(s - a) errs by 3 u |b|, the
// difference from it by less than u |b|). lo2's roundings, at most u K^2 <= 1.4e-12 of
// u (|lo| at the start + sum |t|) over K <= 112 products, are in TREE_U and begin().
struct Chain {
  double hi = 0.0, lo = 0.0, lo2 = 0.0;
};
template <bool R>
__device__ __forceinline__ dd chain_value(const Chain& a, double& r) {
  const dd h = two_sum(a.hi, a.lo);
  const double w = h.lo + a.lo2;
  if constexpr (R) r = fma(fabs(w) > fabs(h.hi) ? 5.0 * CERT_U : CERT_U, fabs(w), r);
  return fast_two_sum(h.hi, w);
}
__device__ __forceinline__ double chain_add(Chain& a, double p, double e) {
  const dd s = two_sum(a.hi, p);
  const double t = s.lo + e;
  const dd z = two_sum(a.lo, t);
  a.hi = s.hi;
  a.lo = z.hi;
  a.lo2 += z.lo;
  return t;
}
template <bool R>
__device__ __forceinline__ void dd_mac(Chain& acc, dd x, dd y, double& r) {
  const double p = x.hi * y.hi;
  const double f = fma(x.hi, y.lo, fma(x.hi, y.hi, -p));
  const double e = fma(x.lo, y.hi, f);
  const double t = chain_add(acc, p, e);
  if constexpr (R) r += fma(fabs(x.lo), fabs(y.lo), TREE_U * ((fabs(f) + fabs(e)) + fabs(t)));
}
template <bool R>
__device__ __forceinline__ void dd_mac_d(Chain& acc, double x, dd y, double& r) {  // x a plain double
  const double p = x * y.hi;
  const double e = fma(x, y.lo, fma(x, y.hi, -p));
  const double t = chain_add(acc, p, e);
  if constexpr (R) r = fma(TREE_U, fabs(e) + fabs(t), r);
}
struct ChainC {
  Chain re, im;
};
__device__ __forceinline__ double tree_abs(ddc z) { return tree_abs(cdd_mag(z.re), cdd_mag(z.im)); }
template <bool R>
__device__ __forceinline__ ddc chain_value(const ChainC& a, double& r) {
  const dd re = chain_value<R>(a.re, r);
  return ddc{re, chain_value<R>(a.im, r)};
}
__device__ __forceinline__ dd dd_signed(dd a, double s) { return dd{s * a.hi, s * a.lo}; }
__device__ __forceinline__ dd swap_pair_dd(dd a) { return dd{swap_pair_d(a.hi), swap_pair_d(a.lo)}; }

// dd_add / dd_mul_d of one component, the operation's own error added to e
template <bool CERT>
__device__ __forceinline__ dd tree_add(dd a, dd b, double& e) {
  if constexpr (!CERT) return dd_add(a, b);
  double o;
  const dd r = cdd_add(a, b, &o);
  e += o;
  return r;
}
template <bool CERT>
__device__ __forceinline__ dd tree_mul_d(dd a, double b, double& e) {
  if constexpr (!CERT) return dd_mul_d(a, b);
  double o;
  const dd r = cdd_mul_d(a, b, &o);
  e += o;
  return r;
}

template <int PM, bool CERT, int... Ps>
__device__ __forceinline__ void tree_row_dd(ChainC& s, double& es, double& r, const cplx& c, const cplx& c2, const ddc (&x)[PM],
                                            const double (&ex)[CERT ? PM : 1], int k1, std::integer_sequence<int, Ps...>) {
  auto term = [&](const cplx& z, int u) __attribute__((always_inline)) {
    dd_mac_d<CERT>(s.re, z.re, x[u].re, r);
    dd_mac_d<CERT>(s.im, z.re, x[u].im, r);
    dd_mac_d<CERT>(s.re, -z.im, x[u].im, r);
    dd_mac_d<CERT>(s.im, z.im, x[u].re, r);
    if constexpr (CERT) es = fma(tree_abs(z), ex[u], es);
  };
  (((Ps < k1) ? (term(row_bcast<(2 * Ps) % 16>(Ps < 8 ? c : c2), 2 * Ps),
                 term(row_bcast<(2 * Ps + 1) % 16>(Ps < 8 ? c : c2), 2 * Ps + 1), 0)
              : 0),
   ...);
}

template <bool LOOP, int H, bool CERT>
__global__ __launch_bounds__(64) void haf_tree_dd_kernel(const cplx* __restrict__ mats, ddc* __restrict__ part,
                                                         double* __restrict__ part_abs) {
  using L = TreeLds<LOOP, H, true>;
  using S = TreeSeries<LOOP, true>;
  constexpr int T2 = TREE_T2, KC = L::KC, KS = L::KS, N = 2 * H, T1 = H - T2, RR = L::RR, PM = L::PM;
  __shared__ ddc lds[L::TOTAL];
  __shared__ double ldse[CERT ? L::TOTAL : 1];  // bounds, at the same places
  dd* const ldc = reinterpret_cast<dd*>(lds);   // components: 2 i, 2 i + 1
  const int lane = threadIdx.x;
  const int64_t b = (int64_t)blockIdx.x >> T1;
  const unsigned p1 = blockIdx.x & ((1u << T1) - 1u);
  const int k1 = __popc(p1);
  const cplx* __restrict__ A = mats + b * N * N;
  auto bound = [&](int i) -> double { return CERT ? ldse[CERT ? i : 0] : 0.0; };

  // ---- leading pairs (haf_tree_kernel), every lane both components
  int ei = 0, ej = 0;
  {
    while (tree_tri(ei + 1, 0) <= lane && ei < 2 * T2) ++ei;
    ej = lane - tree_tri(ei, 0);
  }
  const bool mine = lane < S::ROOT, top = !LOOP && mine && (ei & 1) && ej == ei - 1;
  auto put = [&](int k, ddc v, double e) __attribute__((always_inline)) {
    int o = -1;
    if (k < KC)
      o = lane * KS + k;
    else if (k < H && top)
      o = L::B0 + (ei >> 1);
    if (o >= 0) {
      lds[o] = v;
      if constexpr (CERT) ldse[o] = e;
    }
  };
  if (mine) {
    const int r = PM + ej, i = ei < 2 * T2 ? PM + ei : r;
    put(0, ddc_from((!LOOP && i == r) ? cplx{0.0, 0.0} : A[i * N + r]), 0.0);
  }
  const bool off = p1 == 0 && tree_nonfinite<LOOP, N>(A);
  if (p1 == 0) {
    if (mine) {
      for (int k = 1; k < H; ++k) put(k, ddc_zero(), 0.0);
    }
    if (lane < H) {
      lds[L::S0 + lane] = ddc_zero();
      if constexpr (CERT) ldse[L::S0 + lane] = 0.0;
    }
  } else {
    ddc cur[PM], nxt[PM];
    double ecur[CERT ? PM : 1], enxt[CERT ? PM : 1];
    cplx cr[T1], cr2[PM > 16 ? T1 : 1];
    const int hf = lane >> 5, col = lane & 31;
    const int vcol = col - (32 - RR);
    const bool isv = vcol >= 0, isc = col < 2 * k1;
    int pr[T1];
    int ac = 0, au = 0, au2 = 0;
    {
      unsigned rest = p1;
#pragma unroll
      for (int i = 0; i < T1; ++i) {
        pr[i] = rest ? 2 * __builtin_ctz(rest) : 0;
        rest &= rest - 1;
        if ((col >> 1) == i) ac = pr[i] + (col & 1);
        if (((lane & 15) >> 1) == i) au = pr[i] + (lane & 1);
        if (PM > 16 && 8 + ((lane & 15) >> 1) == i) au2 = pr[i] + (lane & 1);
      }
    }
    if (isv) ac = PM + vcol;
    int vc = L::V0, vn = L::V0 + L::VN;
#pragma unroll
    for (int t = 0; t < PM; ++t) {
      nxt[t] = cur[t] = ddc_zero();
      if constexpr (CERT) enxt[t] = ecur[t] = 0.0;
      if ((t >> 1) < k1) {
        const int r = pr[t >> 1] + ((t & 1) ^ 1);
        const cplx a = A[r * N + ((LOOP && vcol == 2 * T2) ? r : ac)];
        if ((isc || isv) && (LOOP || ac != r)) cur[t] = ddc_from(a);
      }
    }
#pragma unroll
    for (int i = 0; i < T1; ++i) {
      if (i < k1) {
        const int r = pr[i] + 1 - hf;
        cr[i] = (!LOOP && au == r) ? cplx{0.0, 0.0} : A[r * N + au];
        if constexpr (PM > 16) cr2[i] = (!LOOP && au2 == r) ? cplx{0.0, 0.0} : A[r * N + au2];
      }
    }
    if (isv && hf == 0) {
#pragma unroll
      for (int t = 0; t < PM; ++t)
        if ((t >> 1) < k1) {
          lds[vc + t * RR + vcol] = cur[t];
          if constexpr (CERT) ldse[vc + t * RR + vcol] = 0.0;
        }
    }
    constexpr int J = (H + 1) / 2;
#pragma unroll 1
    for (int j = 0; j < J; ++j) {
      {
        double yA[CERT ? PM : 1];
        if constexpr (CERT) {
#pragma unroll
          for (int t = 0; t < PM; ++t) yA[t] = ecur[t];
        }
#pragma unroll
        for (int i = 0; i < T1; ++i)
          if (i < k1) {
            ChainC c;
            double es = TREE_UFL, r = 0.0;
            tree_row_dd<PM, CERT>(c, es, r, cr[i], cr2[PM > 16 ? i : 0], cur, yA, k1, std::make_integer_sequence<int, T1>{});
            const ddc s = chain_value<CERT>(c, r);
            halves_d(s.re.hi, nxt[2 * i].re.hi, nxt[2 * i + 1].re.hi);
            halves_d(s.re.lo, nxt[2 * i].re.lo, nxt[2 * i + 1].re.lo);
            halves_d(s.im.hi, nxt[2 * i].im.hi, nxt[2 * i + 1].im.hi);
            halves_d(s.im.lo, nxt[2 * i].im.lo, nxt[2 * i + 1].im.lo);
            if constexpr (CERT) halves_d(es + r, enxt[2 * i], enxt[2 * i + 1]);
          }
      }
      if (isv && hf == 0) {
#pragma unroll
        for (int t = 0; t < PM; ++t)
          if ((t >> 1) < k1) {
            lds[vn + t * RR + vcol] = nxt[t];
            if constexpr (CERT) ldse[vn + t * RR + vcol] = enxt[t];
          }
      }
      auto term = [&](ChainC& s, double& es, const ddc& x, double ex, const ddc& y, double ey)
                      __attribute__((always_inline)) {
        double r = 0.0;
        dd_mac<CERT>(s.re, x.re, y.re, r);
        dd_mac<CERT>(s.im, x.re, y.im, r);
        dd_mac<CERT>(s.re, dd_neg(x.im), y.im, r);
        dd_mac<CERT>(s.im, x.im, y.re, r);
        if constexpr (CERT) {
          const double Y = tree_abs(y);
          es = fma(tree_abs(x), ey, fma(ex, Y + ey, es + r));
        }
      };
      ChainC pe, po;
      double epe = TREE_UFL, epo = TREE_UFL;
      auto swp = [](const ddc& z) -> ddc { return ddc{swap_pair_dd(z.re), swap_pair_dd(z.im)}; };
#pragma unroll
      for (int i = 0; i < T1; ++i)
        if (i < k1) {
          const int t = 2 * i;
          const ddc y = swp(cur[t + 1]), z = swp(nxt[t + 1]);
          const double ey = CERT ? swap_pair_d(ecur[CERT ? t + 1 : 0]) : 0.0;
          const double ez = CERT ? swap_pair_d(enxt[CERT ? t + 1 : 0]) : 0.0;
          const double ex = CERT ? ecur[CERT ? t : 0] : 0.0, en = CERT ? enxt[CERT ? t : 0] : 0.0;
          term(pe, epe, cur[t], ex, y, ey);
          term(po, epo, cur[t], ex, z, ez);
          term(po, epo, nxt[t], en, y, ey);
        }
      if (isc && hf == 0) {
        const int o = L::PB0 + (2 * j + 1) * PM + col;
        lds[o] = ddc_mul_d(chain_value<CERT>(pe, epe), 2.0);
        if constexpr (CERT) ldse[o] = 2.0 * epe;
        if (2 * j + 2 < H) {
          lds[o + PM] = chain_value<CERT>(po, epo);
          if constexpr (CERT) ldse[o + PM] = epo;
        }
      }
      __syncthreads();
      if (mine || (LOOP && lane == S::ROOT)) {
        ChainC s1, s2;
        double e1 = TREE_UFL, e2 = TREE_UFL;
#pragma unroll 1
        for (int i = 0; i < k1; ++i) {
          const int o = 2 * i * RR;
          const int x0 = vc + o + ei, x1 = x0 + RR, y0 = vc + o + ej, y1 = y0 + RR, z0 = vn + o + ej, z1 = z0 + RR;
          const ddc u0 = lds[x0], u1 = lds[x1];
          term(s1, e1, u0, bound(x0), lds[y1], bound(y1));
          term(s1, e1, u1, bound(x1), lds[y0], bound(y0));
          term(s2, e2, u0, bound(x0), lds[z1], bound(z1));
          term(s2, e2, u1, bound(x1), lds[z0], bound(z0));
        }
        const ddc v1 = chain_value<CERT>(s1, e1), v2 = chain_value<CERT>(s2, e2);
        if (LOOP && lane == S::ROOT) {
          lds[L::E0 + 2 * j] = v1;
          lds[L::E0 + 2 * j + 1] = v2;
          if constexpr (CERT) {
            ldse[L::E0 + 2 * j] = e1;
            ldse[L::E0 + 2 * j + 1] = e2;
          }
        } else {
          put(2 * j + 1, v1, e1);
          put(2 * j + 2, v2, e2);
        }
      }
      __syncthreads();
#pragma unroll
      for (int t = 0; t < PM; ++t) {
        cur[t] = nxt[t];
        if constexpr (CERT) ecur[t] = enxt[t];
      }
      const int sw = vc;
      vc = vn;
      vn = sw;
    }
    if (lane < H) {
      ddc s = ddc_zero();
      double e = TREE_UFL;
      auto add = [&](const ddc& x, double ex) __attribute__((always_inline)) {
        e += ex;
        s = ddc{tree_add<CERT>(s.re, x.re, e), tree_add<CERT>(s.im, x.im, e)};
      };
      if (lane == 0) {
        for (unsigned rest = p1; rest; rest &= rest - 1) {
          const int t = 2 * __builtin_ctz(rest);
          add(ddc_from(A[t * N + t + 1]), 0.0);
          add(ddc_from(A[(t + 1) * N + t]), 0.0);
        }
      } else {
        for (int i = 0; i < 2 * k1; ++i) add(lds[L::PB0 + lane * PM + i], bound(L::PB0 + lane * PM + i));
      }
      s = ddc_mul_d(s, 0.5);
      e = fma(0.5, e, TREE_UFL);
      if constexpr (LOOP) {
        const double f = 0.5 * (lane + 1);
        const ddc x = lds[L::E0 + lane];
        double ex = f * bound(L::E0 + lane);
        const ddc y{tree_mul_d<CERT>(x.re, f, ex), tree_mul_d<CERT>(x.im, f, ex)};
        add(y, ex);
      }
      lds[L::S0 + lane] = s;
      if constexpr (CERT) ldse[L::S0 + lane] = e;
    }
  }
  __syncthreads();

  // ---- the tree. This lane's component: 0 real, 1 imaginary; its part of x y is
  // x.re y[half] + (half ? x.im : -x.im) y[1 - half].
  const int half = lane & 1;
  const double sgi = half ? 1.0 : -1.0;
  // a0, a1 += coefficients d, d + 1 of sx x y, series at xo, yo (a1 only with TWO;
  // LATE: without its product x_0 y_(d+1)); the bounds' share in e0, e1, the
  // roundings' in r0, r1. The next operands load while the present ones are used.
  struct Acc {
    Chain v;
    double e = TREE_UFL, r = 0.0;
  };
  auto conv = [&](auto two_, auto late_, int xo, int yo, int d, double sx, Acc& a0, Acc& a1)
                  __attribute__((always_inline)) {
    constexpr bool TWO = decltype(two_)::value, LATE = decltype(late_)::value;
    dd p0{0.0, 0.0}, p1v{0.0, 0.0};
    double yp = 0.0, yq = 0.0;
    if constexpr (TWO && !LATE) {
      p0 = ldc[2 * (yo + d + 1) + half];
      p1v = ldc[2 * (yo + d + 1) + 1 - half];
      if constexpr (CERT) {
        const double Y = tree_abs(cdd_mag(p0), cdd_mag(p1v)), ey = ldse[yo + d + 1];
        yp = ey;
        yq = Y + ey;
      }
    }
    dd x0 = ldc[2 * xo], x1 = ldc[2 * xo + 1], m0 = ldc[2 * (yo + d) + half], m1 = ldc[2 * (yo + d) + 1 - half];
    double xe = bound(xo), me = bound(yo + d);
#pragma unroll 2
    for (int i = 0; i <= d; ++i) {
      const dd xr = dd_signed(x0, sx), xi = dd_signed(x1, sx * sgi), n0 = m0, n1 = m1;
      const double ex = xe, ey = me;
      const int in = TWO || i < d ? i + 1 : i, jn = i < d ? d - i - 1 : 0;
      x0 = ldc[2 * (xo + in)];
      x1 = ldc[2 * (xo + in) + 1];
      m0 = ldc[2 * (yo + jn) + half];
      m1 = ldc[2 * (yo + jn) + 1 - half];
      xe = bound(xo + in);
      me = bound(yo + jn);
      dd_mac<CERT>(a0.v, xr, n0, a0.r);
      if constexpr (TWO) dd_mac<CERT>(a1.v, xr, p0, a1.r);
      dd_mac<CERT>(a0.v, xi, n1, a0.r);
      if constexpr (TWO) dd_mac<CERT>(a1.v, xi, p1v, a1.r);
      p0 = n0;
      p1v = n1;
      if constexpr (CERT) {
        const double X = tree_abs(cdd_mag(xr), cdd_mag(xi)), Y = tree_abs(cdd_mag(n0), cdd_mag(n1));
        a1.e = fma(X, yp, fma(ex, yq, a1.e));
        yp = ey;
        yq = Y + ey;
        a0.e = fma(X, yp, fma(ex, yq, a0.e));
      }
    }
    if constexpr (TWO) {
      const dd xr = dd_signed(x0, sx), xi = dd_signed(x1, sx * sgi);
      dd_mac<CERT>(a1.v, xr, p0, a1.r);
      dd_mac<CERT>(a1.v, xi, p1v, a1.r);
      if constexpr (CERT) a1.e = fma(tree_abs(cdd_mag(xr), cdd_mag(xi)), yp, fma(xe, yq, a1.e));
    }
  };
  using Yes = std::true_type;
  using No = std::false_type;
  // closes a chain: its errors in both components join the bound
  auto close = [&](Acc& a) __attribute__((always_inline)) -> dd {
    const dd v = chain_value<CERT>(a.v, a.r);
    if constexpr (CERT) a.e += tree_abs(a.r, swap_pair_d(a.r));
    return v;
  };
  auto begin = [](Acc& a, dd v) __attribute__((always_inline)) {
    a.v.hi = v.hi;
    a.v.lo = v.lo;
    if constexpr (CERT) a.r = 1e-11 * CERT_U * fabs(v.lo);
  };
  // e + the errors of both components' operations since r was zero
  auto both = [&](double e, double r) -> double { return CERT ? e + tree_abs(r, swap_pair_d(r)) : 0.0; };
#pragma unroll 1
  for (int l = 0; l < T2; ++l) {
    const TreeTask k = tree_table<LOOP, true>.t[l][lane & ~1], kb = tree_table<LOOP, true>.t[l][lane | 1];
    const bool on = k.flags & TREE_ON, isq = k.flags & TREE_PIVOT;
    const int vo = isq ? L::S0 + k.sc * H : k.w * KS;  // the task's series
    // right-hand sides: P = b (m = -2) for the pivot, the second lane's y operand (m = 1) for rows
    if (on) {
      const double m = isq ? -2.0 : 1.0;
      const int po = (isq ? k.px : kb.py) * KS;
      // coefficient d of m P, where its chain starts
      auto first = [&](Acc& a, int d) __attribute__((always_inline)) {
        const int o = d < KC ? po + d : L::B0 + k.b;
        begin(a, dd_signed(ldc[2 * o + half], m));
        if constexpr (CERT) a.e = fma(fabs(m), ldse[o], TREE_UFL);
      };
      auto rhs = [&](int d, dd z, double e) __attribute__((always_inline)) {
        if (isq) {
          if (d < KC) {
            ldc[2 * (k.q * KS + d) + half] = z;
            if constexpr (CERT) ldse[k.q * KS + d] = e;
          }
          const double f = -0.5 * (d + 1);
          double r = 0.0;
          z = tree_mul_d<CERT>(z, f, r);
          e = both(-f * e, r);
        }
        if (isq || d < KC) {
          ldc[2 * (vo + d) + half] = z;
          if constexpr (CERT) ldse[vo + d] = e;
        }
      };
      Acc a;
      first(a, 0);
      rhs(0, dd{a.v.hi, a.v.lo}, a.e);
#pragma unroll 1
      for (int d = 0; d < H - 1; d += 2) {
        Acc a0, a1;
        first(a0, d + 1);
        if (d + 1 < H - 1) {
          first(a1, d + 2);
          conv(Yes{}, No{}, k.px * KS, k.py * KS, d, 1.0, a0, a1);
          conv(Yes{}, No{}, kb.px * KS, kb.py * KS, d, -1.0, a0, a1);
        } else {
          conv(No{}, No{}, k.px * KS, k.py * KS, d, 1.0, a0, a1);
          conv(No{}, No{}, kb.px * KS, kb.py * KS, d, -1.0, a0, a1);
        }
        const dd s0 = close(a0), s1 = close(a1);
        rhs(d + 1, s0, a0.e);
        if (d + 1 < H - 1) rhs(d + 2, s1, a1.e);
      }
    }
    __syncthreads();
    // q y = rhs in place, two coefficients at a time (the partner lane's component
    // of the earlier ones comes through LDS)
    const int nrec = isq ? H : KC, qo = k.q * KS;
    auto start = [&](Acc& a, int o) __attribute__((always_inline)) {
      begin(a, ldc[2 * o + half]);
      if constexpr (CERT) a.e = ldse[o];
    };
#pragma unroll 1
    for (int d = 1; d < H; d += 2) {
      Acc a0, a1;
      const bool two = d + 1 < nrec;
      if (on && d < nrec) {
        start(a0, vo + d);
        if (two) {
          start(a1, vo + d + 1);
          conv(Yes{}, Yes{}, qo, vo, d - 1, -1.0, a0, a1);
        } else {
          conv(No{}, No{}, qo, vo, d - 1, -1.0, a0, a1);
        }
        ldc[2 * (vo + d) + half] = close(a0);
        if constexpr (CERT) ldse[vo + d] = a0.e;
      }
      __syncthreads();
      if (on && two) {
        conv(No{}, No{}, qo, vo + d, 0, -1.0, a1, a0);
        ldc[2 * (vo + d + 1) + half] = close(a1);
        if constexpr (CERT) ldse[vo + d + 1] = a1.e;
      }
      __syncthreads();
    }
    if (on && isq) {  // the child's sigma (at the last level the include leaf's)
#pragma unroll 1
      for (int d = 0; d < H; ++d) {
        const dd x = ldc[2 * (L::S0 + k.sp * H + d) + half], y = ldc[2 * (vo + d) + half];
        double r = 0.0;
        ldc[2 * (vo + d) + half] = tree_add<CERT>(x, y, r);
        if constexpr (CERT) ldse[vo + d] = both(bound(L::S0 + k.sp * H + d) + ldse[vo + d], r);
      }
    }
    __syncthreads();
    if (k.flags & TREE_ENTRY) {
      // kb: the second product's factors
      const bool isE = k.flags & TREE_E;
      if (!isE) {
        ldc[2 * (k.ed * KS) + half] = ldc[2 * (k.ez * KS) + half];
        if constexpr (CERT) ldse[k.ed * KS] = ldse[k.ez * KS];
      }
      // coefficient d of the product: a share of sigma, or added to coefficient d + 1
      auto first = [&](Acc& a, int d) __attribute__((always_inline)) {
        if (!isE && d + 1 < H) {
          const int o = d + 1 < KC ? k.ez * KS + d + 1 : L::B0 + k.zb;
          begin(a, ldc[2 * o + half]);
          if constexpr (CERT) a.e += ldse[o];
        }
      };
      auto out = [&](int d, dd s, double e) __attribute__((always_inline)) {
        if (isE) {
          const int o = L::S0 + k.esc * H + d;
          const double f = 0.5 * (d + 1);
          double r = 0.0;
          const dd x = tree_mul_d<CERT>(s, f, r), z = ldc[2 * o + half];
          ldc[2 * o + half] = tree_add<CERT>(z, x, r);
          if constexpr (CERT) ldse[o] = both(fma(f, e, ldse[o]), r);
        } else if (d + 1 < H) {
          const int t = d + 1 < KC ? k.ed * KS + d + 1 : L::B0 + k.db;  // TREE_BX: a slot nothing reads
          if constexpr (CERT) ldse[t] = e;
          ldc[2 * t + half] = s;
        }
      };
#pragma unroll 1
      for (int d = 0; d < KC; d += 2) {
        Acc a0, a1;
        first(a0, d);
        if (d + 1 < KC) {
          first(a1, d + 1);
          conv(Yes{}, No{}, k.et * KS, k.ew * KS, d, 1.0, a0, a1);
          conv(Yes{}, No{}, kb.et * KS, kb.ew * KS, d, 1.0, a0, a1);
        } else {
          conv(No{}, No{}, k.et * KS, k.ew * KS, d, 1.0, a0, a1);
          conv(No{}, No{}, kb.et * KS, kb.ew * KS, d, 1.0, a0, a1);
        }
        const dd s0 = close(a0), s1 = close(a1);
        out(d, s0, a0.e);
        if (d + 1 < KC) out(d + 1, s1, a1.e);
      }
    }
    __syncthreads();
  }
  // ---- Newton: lane pair i on leaf i (node i / 2; even: included), coefficients
  // e_1 .. e_H of leaf i over the matrices (free now)
  const int nu = lane >> 2, incl = ((lane >> 1) & 1) ^ 1;
  const bool live = lane < 4 << (T2 - 1);
  int slot = 0;
  if (incl) {
    slot = (1 << (T2 - 1)) + nu;
  } else if (nu) {
    const int p = __builtin_ctz((unsigned)nu);
    slot = (1 << (T2 - 2 - p)) + (nu >> (p + 1));
  }
  const int so = L::S0 + (live ? slot : 0) * H, eo = (lane >> 1) * H;
  static_assert((2 << (T2 - 1)) * H <= S::Q * KS, "Newton scratch");
  dd coeff{0.0, 0.0};
  double ecoeff = 0.0;
#pragma unroll 1
  for (int j = 1; j <= H; ++j) {
    if (live) {
      Acc a, none;
      begin(a, ldc[2 * (so + j - 1) + half]);  // sigma_j e_0
      if constexpr (CERT) a.e += ldse[so + j - 1];
      if (j > 1) conv(No{}, No{}, so, eo, j - 2, 1.0, a, none);
      const dd s = close(a);
      const double e = a.e;
      if constexpr (CERT) {
        double r;
        coeff = cdd_div_d(s, (double)j, &r);
        ecoeff = e / (double)j + tree_abs(r, swap_pair_d(r));
        ldse[eo + j - 1] = ecoeff;
      } else {
        coeff = dd_div_d(s, (double)j);
      }
      ldc[2 * (eo + j - 1) + half] = coeff;
    }
    __syncthreads();
  }
  if (!live) {
    coeff = dd{0.0, 0.0};
    ecoeff = 0.0;
  }
  if ((H - (k1 + __popc((unsigned)nu) + incl)) & 1) coeff = dd_neg(coeff);
  // sum over the leaves: lanes of equal parity
#pragma unroll
  for (int m = 2; m < 64; m <<= 1) {
    const dd o{shfl_xor_d(coeff.hi, m), shfl_xor_d(coeff.lo, m)};
    if constexpr (CERT) {
      double r;
      const double oe = shfl_xor_d(ecoeff, m);
      coeff = cdd_add(coeff, o, &r);
      ecoeff = ecoeff + oe + tree_abs(r, swap_pair_d(r));
    } else {
      coeff = dd_add(coeff, o);
    }
  }
  if (lane < 2) {
    reinterpret_cast<dd*>(part)[2 * (int64_t)blockIdx.x + lane] = off ? dd{NAN, NAN} : coeff;
    if constexpr (CERT) {
      if (lane == 0) part_abs[blockIdx.x] = off ? INFINITY : cert_finish(ecoeff, TREE_DEPTH);
    }
  }
}

}  // namespace gbsk
