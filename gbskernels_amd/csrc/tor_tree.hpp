// tor_tree.hpp -- real-domain torontonian of 6 or more modes: one wave per
// (instance, include pattern of the leading modes). Included by tor.hip, which
// defines the arithmetic policies, the split and the per-lane trailing walk.
//
// Same subset tree and the same operations in the same order as the general
// workgroup of tor.hip (values and bounds are those bits); what differs is where
// the matrices live:
//  * leading modes: lane c holds column c of the active matrix in registers, so
//    a pivot step is one product, one lane broadcast and one fma a row, with no
//    LDS traffic and no barrier (in LDS: four reads, a write and index work an
//    entry);
//  * middle modes 0..3: breadth first over include children in LDS, in 2 x 2
//    blocks (x, p of one mode against x, p of another) with the modes in reverse
//    order: excluding a mode keeps a prefix of its parent's blocks, so every
//    address is a node's base plus a constant, and a task is one block (eight
//    fma, seven 16-byte reads);
//  * middle modes 4 and 5: each lane eliminates them on its own copy (lane k =
//    leaf k of the six-mode tree), so the two widest levels never enter LDS:
//    18.5 KB instead of 29 KB at 11 modes, 8 waves a CU, the number its
//    registers allow;
//  * trailing modes: bottom_walk, unchanged.
// The general workgroup spent most of its time above the trailing walk (LDS
// latency of the leading steps, index work of the middle ones). Measured on
// MI355X, general workgroup -> this kernel, B = 4096: fp64 8 / 12 / 16 modes 33.5 /
// 206 / 3136 -> 21.7 / 101 / 1391 us, certified 8 / 12 81 / 560 -> 41 / 294 us, dd 8 / 12
// 135 / 1492 -> 66 / 1115 us; faster at every count from 6 to 20 modes and every
// tier. What bounds it: FP64 issue of the trailing walk (about 1500 of the 3400
// instructions a wave runs at 16 modes) at two waves a SIMD.
#pragma once

namespace gbsk {

constexpr int TREE_LDS_LEVELS = 4;  // middle modes walked in LDS; the other two in registers

// lane `src`'s value in every lane (src wave-uniform)
__device__ __forceinline__ double lane_bcast(double v, int src) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, src);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), src);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ dd lane_bcast(dd v, int src) { return dd{lane_bcast(v.hi, src), lane_bcast(v.lo, src)}; }
__device__ __forceinline__ cv lane_bcast(cv v, int src) { return cv{lane_bcast(v.v, src), lane_bcast(v.e, src)}; }
__device__ __forceinline__ cdd lane_bcast(cdd v, int src) { return cdd{lane_bcast(v.v, src), lane_bcast(v.e, src)}; }

// 2 x 2 blocks of a matrix of m modes: block (I, J), I >= J (reversed modes), at
// 4 tri(I, J); element [s][t] is row t of mode J against column s of mode I (in
// the original order mode J comes after I). A diagonal block's [1][0] is unused.
__host__ __device__ constexpr int blocks_size(int m) { return 2 * m * (m + 1); }
// first entry of level lv's include matrices (2^(lv-1) of base - lv modes)
__host__ __device__ constexpr int tree_region_at(int base, int lv) {
  if (lv == 0) return 0;
  int r = blocks_size(base);
  for (int d = 1; d < lv; ++d) r += (1 << (d - 1)) * blocks_size(base - d);
  return r;
}

// Reversed mode M_ - 1 of a matrix of M_ modes eliminated by one lane: N (LDS or
// registers) holds it, Y receives the first M_ - 1 modes. A lane that excludes
// the mode copies them: its multipliers are zero (a product with zero leaves
// every bit; a row that is not finite makes the including lane's pivots fail, so
// the instance is off anyway), or, where a bound would still be charged for the
// step, it takes no step.
template <class Ar, int M_, class T>
__device__ __forceinline__ void lane_include(const T* N, T* Y, bool inc, bool& bad, T& det) {
  constexpr int p = M_ - 1, P0 = 4 * tri(p, p), Q0 = 4 * tri(p, 0), W = p > 0 ? 2 * p : 1;
  const T a = N[P0], b01 = N[P0 + 1];
  const T ra = Ar::recip(a);
  const T c = Ar::sub(N[P0 + 3], Ar::mul(Ar::mul(b01, b01), ra));
  const T rc = Ar::recip(c);
  bad |= !Ar::pos(a) || !Ar::pos(c);
  if (inc) det = Ar::mul(det, Ar::mul(a, c));
  T x0[W], x1[W], l0[W], l1[W];
  auto each = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
    for (int I = 0; I < p; ++I)
#pragma unroll
      for (int J = 0; J <= I; ++J)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (I != J || q != 2) f(4 * tri(I, J) + q, 2 * I + (q >> 1), 2 * J + (q & 1));
  };
  if constexpr (Ar::CERT) each([&](int e, int, int) __attribute__((always_inline)) { Y[e] = N[e]; });
  if (!Ar::CERT || inc) {
#pragma unroll
    for (int J = 0; J < p; ++J)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int r = 2 * J + t;
        x0[r] = N[Q0 + 4 * J + t];
        l0[r] = Ar::mul(x0[r], ra);
        x1[r] = Ar::fms(l0[r], b01, N[Q0 + 4 * J + 2 + t]);
        l1[r] = Ar::mul(x1[r], rc);
        if constexpr (!Ar::CERT) {
          l0[r] = inc ? l0[r] : Ar::zero();
          l1[r] = inc ? l1[r] : Ar::zero();
        }
      }
    each([&](int e, int i, int j) __attribute__((always_inline)) {
      Y[e] = Ar::fms(l1[j], x1[i], Ar::fms(l0[j], x0[i], Ar::CERT ? Y[e] : N[e]));
    });
  }
}

// fp64 and dd run two waves per SIMD (their LDS allows 8 and 7 a CU). dd at three
// trailing modes then spills 63 VGPRs to scratch, mostly the leading columns, and
// is still faster than one wave with 62 AGPRs: 10 / 12 / 14 modes (B = 4096 / 4096 /
// 3051) 280 / 1298 / 4369 -> 249 / 1115 / 3636 us. The certified policies need 512
// registers: one wave.
template <class Ar>
constexpr int tor_tree_waves() { return std::is_same<Ar, RF64>::value || std::is_same<Ar, RDD>::value ? 2 : 1; }

// t_k = read(k) for k < N, a barrier, then write(k, t_k): no array (it went to scratch)
template <int N, class Rd, class Wr>
__device__ __forceinline__ void read_then_write(const Rd& read, const Wr& write) {
  const auto t = read(N - 1);
  if constexpr (N > 1)
    read_then_write<N - 1>(read, write);
  else
    __syncthreads();
  write(N - 1, t);
}

// Certified dd keeps up to 11 leading modes in LDS, one entry of the active block a
// lane and step (eliminate, tor.hip): a step of its arithmetic is some 100 operations,
// and one column a lane leaves 64 - D lanes idle, 2.8 times the steps at 10 leading
// modes and no trailing ones. General workgroup / one column a lane / this, us: one instance
// over the device at 12 / 16 / 18 modes 83 / 102 / 83, 126 / 155 / 125, 169 / 192 / 161, one of a batch at
// 18 modes 149 / 169 / 136, B = 4096 at 12 / 16 modes 4235 / 3493 / 2993, 78300 / 66100 / 53700. Without
// leading modes LM is 0 (their LDS cost a third of the waves: 8 modes, B = 1024 48 -> 60 us).
template <class Ar, int LM>
constexpr bool tor_lead_lds() { return std::is_same<Ar, RCDD>::value && LM > 0 && LM <= 11; }

// LM: leading modes the register columns have room for.
template <class Ar, int R, bool KAPPA, int LM>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(tor_tree_waves<Ar>()))) void tor_tree_kernel(
    const cplx* __restrict__ mats, int T1, typename Ar::P* __restrict__ part, double* __restrict__ part_abs,
    const TorDirect dir) {
  using T = typename Ar::T;
  static_assert(Ar::SYM && Ar::TASK_REGS, "symmetric register-task policies");
  constexpr int BASE = TOR_T2 + R, DB = 2 * BASE;
  constexpr int LV = TREE_LDS_LEVELS, MT = BASE - LV;  // MT modes left where the lanes take over
  static_assert(TOR_T2 == LV + 2 && DB + 2 * LM <= 64, "two middle modes in registers, one column a lane");
  constexpr bool LEAD_LDS = tor_lead_lds<Ar, LM>();
  constexpr int LEVN = tree_region_at(BASE, LV + 1), WN = LEAD_LDS ? (DB + 2 * LM) * (DB + 2 * LM) : 0;
  __shared__ T lev[LEVN > WN ? LEVN : WN];
  __shared__ T bdet[(2 << LV) - 1];  // determinants, level d node n at 2^d - 1 + n
  __shared__ unsigned short bij[(BASE * (BASE - 1)) / 2];
  const int lane = threadIdx.x;
  const int nm = BASE + T1, dim = 2 * nm;
  const int64_t wg = blockIdx.x, b = wg >> T1;
  const unsigned p1 = (unsigned)(wg & ((1ll << T1) - 1));
  const int k1 = __popc(p1);
  for (int e = lane; e < BASE * (BASE - 1) / 2; e += 64) {  // (I, J) of every block a level forms
    int i, j;
    tri_decode(e, i, j);
    bij[e] = (unsigned short)(i << 8 | j);
  }

  // ---- A = I - O on the active modes (the trailing BASE modes, then the
  // included leading ones), mode-major: lane c holds column c, X[r] row r. Only
  // active entries are read; the workgroup with every leading mode included
  // reads all of O, so a complex entry anywhere still flags the instance.
  bool bad = false;
  T det = Ar::one();
  if constexpr (LEAD_LDS) {
    // W: the active block, row-major, included leading modes first
    __shared__ unsigned char amode[BASE + LM];
    T* const W = lev;
    const cplx* O = mats + b * dim * dim;
    const int D = DB + 2 * k1;
    if (lane < BASE + k1) {
      unsigned rest = p1;
      for (int i = 0; i < lane && rest; ++i) rest &= rest - 1;
      amode[lane] = (unsigned char)(lane < k1 ? __builtin_ctz(rest) : T1 + lane - k1);
    }
    __syncthreads();
    for (int e = lane; e < D * D; e += 64) {
      const int r = e / D, c = e - r * D;
      const cplx o = O[(amode[r >> 1] + (r & 1) * nm) * dim + amode[c >> 1] + (c & 1) * nm];
      W[e] = r == c ? Ar::one_minus(o) : Ar::neg(o);
      bad |= !Ar::domain(o);
    }
    __syncthreads();
#pragma unroll 1
    for (int q = 0; q < k1; ++q) {
      const T a = eliminate<Ar>(W, D, 2 * q);
      const T c = eliminate<Ar>(W, D, 2 * q + 1);
      bad |= !Ar::pos(a) || !Ar::pos(c);
      det = Ar::mul(det, Ar::mul(a, c));
    }
    // level 0 in place: read everything, then write
    constexpr int N0 = DB * (DB + 1) / 2, PER = (N0 + 63) / 64;
    read_then_write<PER>(
        [&](int k) __attribute__((always_inline)) {
          int i = 0, j = 0;
          if (lane + 64 * k < N0) tri_decode(lane + 64 * k, i, j);
          return W[(2 * k1 + i) * D + 2 * k1 + j];
        },
        [&](int k, const T& t) __attribute__((always_inline)) {
          if (lane + 64 * k < N0) {
            int i, j;
            tri_decode(lane + 64 * k, i, j);
            const int I = BASE - 1 - (j >> 1);
            lev[2 * I * (I + 1) + 2 * (j & 1) + 4 * (BASE - 1 - (i >> 1)) + (i & 1)] = t;
          }
        });
  } else {
    T X[DB + 2 * LM];
    {
      const cplx* O = mats + b * dim * dim;
      int mc = T1 + (lane >> 1);
      if (lane >= DB) {
        mc = 0;
        unsigned rest = p1;
        const int q = (lane - DB) >> 1;
        for (int i = 0; i < q; ++i) rest &= rest - 1;
        if (rest) mc = __builtin_ctz(rest);
      }
      const bool on = lane < DB + 2 * k1;
      const int gc = on ? mc + (lane & 1) * nm : 0;
      cplx raw[DB + 2 * LM];
#pragma unroll
      for (int r = 0; r < DB; ++r) raw[r] = O[(T1 + (r >> 1) + (r & 1) * nm) * dim + gc];
      unsigned rest = p1;
#pragma unroll
      for (int q = 0; q < LM; ++q) {
        raw[DB + 2 * q] = raw[DB + 2 * q + 1] = cplx{0.0, 0.0};
        if (q < k1) {
          const int m = __builtin_ctz(rest);
          rest &= rest - 1;
          raw[DB + 2 * q] = O[m * dim + gc];
          raw[DB + 2 * q + 1] = O[(m + nm) * dim + gc];
        }
      }
#pragma unroll
      for (int r = 0; r < DB + 2 * LM; ++r) {
        X[r] = r == lane ? Ar::one_minus(raw[r]) : Ar::neg(raw[r]);
        bad |= on && !Ar::domain(raw[r]);
      }
    }

    // ---- eliminate the included leading modes (mode order, x then p pivot): the
    // pivot mode's rows are X[DB], X[DB + 1]; the rows above move down after it
#pragma unroll 1
    for (int q = 0; q < k1; ++q) {
      T piv[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int src = DB + 2 * q + t;
        piv[t] = lane_bcast(X[DB + t], src);
        const T rp = Ar::recip(piv[t]);
        auto step = [&](int r) __attribute__((always_inline)) {
          X[r] = Ar::fms(lane_bcast(Ar::mul(X[r], rp), src), X[DB + t], X[r]);
        };
#pragma unroll
        for (int r = 0; r < DB; ++r) step(r);
        if (t == 0) step(DB + 1);
#pragma unroll
        for (int i = 1; i < LM; ++i)
          if (q + i < k1) {
            step(DB + 2 * i);
            step(DB + 2 * i + 1);
          }
      }
      bad |= !Ar::pos(piv[0]) || !Ar::pos(piv[1]);
      det = Ar::mul(det, Ar::mul(piv[0], piv[1]));
#pragma unroll
      for (int r = DB; r + 2 < DB + 2 * LM; ++r) X[r] = X[r + 2];
    }
    // level 0: the lower triangle (row r >= column = lane) in reversed blocks
    {
      const int I = BASE - 1 - (lane >> 1);
      T* const row = lev + 2 * I * (I + 1) + 2 * (lane & 1);
      if (lane < DB) {
#pragma unroll
        for (int r = 0; r < DB; ++r)
          if (r >= lane) row[4 * (BASE - 1 - (r >> 1)) + (r & 1)] = X[r];
      }
    }
  }
  if (lane == 0) bdet[0] = det;
  __syncthreads();

  // ---- middle modes 0..3: node n of level d (pattern bits, first mode most
  // significant) reads the matrix its last include formed
  auto node_at = [&](int d, int n) __attribute__((always_inline)) {
    if (n == 0) return 0;
    const int p = __builtin_ctz((unsigned)n), lv = d - p, g = n >> (p + 1);
    int r = 0;
#pragma unroll
    for (int i = 1; i <= LV; ++i)
      if (lv == i) r = tree_region_at(BASE, i) + g * blocks_size(BASE - i);
    return r;
  };
#pragma unroll
  for (int d = 0; d < LV; ++d) {
    const int m = BASE - d, p = m - 1, P0 = 4 * tri(p, p), Q0 = 4 * tri(p, 0);
    // pivots and reduced second rows, one (node, mode) a lane. The pivot's row
    // of blocks is read by this node alone: the reduced row and the reciprocals
    // take its place
    {
      const int n = lane / p, J = lane - n * p;
      const bool on = n < (1 << d);
      T* const N = lev + (on ? node_at(d, n) : 0);
      const T a = N[P0], b01 = N[P0 + 1];
      const T ra = Ar::recip(a);
      const T c = Ar::sub(N[P0 + 3], Ar::mul(Ar::mul(b01, b01), ra));
      const T rc = Ar::recip(c);
      const T x0 = Ar::fms(Ar::mul(N[Q0 + 4 * J], ra), b01, N[Q0 + 4 * J + 2]);
      const T x1 = Ar::fms(Ar::mul(N[Q0 + 4 * J + 1], ra), b01, N[Q0 + 4 * J + 3]);
      __syncthreads();
      if (on) {
        N[Q0 + 4 * J + 2] = x0;
        N[Q0 + 4 * J + 3] = x1;
        if (J == 0) {
          N[P0 + 2] = ra;
          N[P0 + 3] = rc;
          bad |= !Ar::pos(a) || !Ar::pos(c);
          const T dn = bdet[(1 << d) - 1 + n];
          bdet[(2 << d) - 1 + 2 * n] = dn;
          bdet[(2 << d) - 1 + 2 * n + 1] = Ar::mul(dn, Ar::mul(a, c));
        }
      }
    }
    __syncthreads();
    // include children, one block a task
    const int NB = tri(p, 0), total = NB << d;
    T* const Y = lev + tree_region_at(BASE, d + 1);
#pragma unroll 1
    for (int idx = lane; idx < total; idx += 64) {
      const int n = idx / NB, e = idx - n * NB;
      const int ij = bij[e], I = ij >> 8, J = ij & 255;
      const T* const N = lev + node_at(d, n);
      const T ra = N[P0 + 2], rc = N[P0 + 3];
      const T* const xi = N + Q0 + 4 * I;
      const T* const xj = N + Q0 + 4 * J;
      const T* const src = N + 4 * e;
      const T l0[2] = {Ar::mul(xj[0], ra), Ar::mul(xj[1], ra)};
      const T l1[2] = {Ar::mul(xj[2], rc), Ar::mul(xj[3], rc)};
      T v[4];
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          v[2 * s + t] = Ar::fms(l1[t], xi[2 + s], Ar::fms(l0[t], xi[s], src[2 * s + t]));
      T* const dst = Y + 4 * idx;
#pragma unroll
      for (int s = 0; s < 4; ++s) dst[s] = v[s];
    }
    __syncthreads();
  }

  // ---- middle modes 4 and 5, then the trailing modes, in registers
  const int n4 = lane >> 2;
  T my_det = bdet[(1 << LV) - 1 + n4];
  T M[blocks_size(MT - 1)], M5[R > 0 ? blocks_size(R) : 1];
  lane_include<Ar, MT>(lev + node_at(LV, n4), M, (lane >> 1) & 1, bad, my_det);
  lane_include<Ar, MT - 1>(M, M5, lane & 1, bad, my_det);
  constexpr int SLOT = tor_slot<Ar, R>();
  T task[SLOT > 0 ? SLOT : 1];  // packed lower triangle, original mode order
#pragma unroll
  for (int e = 0; e < SLOT; ++e) {
    const int r = tri_row(e), c = tri_col(e);
    task[e] = M5[4 * tri(R - 1 - (c >> 1), R - 1 - (r >> 1)) + 2 * (c & 1) + (r & 1)];
  }
  T acc = Ar::zero();
  double aacc = 0.0;
  bottom_walk<Ar, R>(task, my_det, k1 + __popc((unsigned)lane), nm, bad, acc, aacc);
  const bool off = __any(bad);
  acc = Ar::sum64(acc);
  if (KAPPA) aacc = group_sum<64>(aacc);
  if (lane == 0) tor_store<Ar, KAPPA, false>(acc, aacc, off, b, p1, T1, part, part_abs, dir);
}

}  // namespace gbsk
