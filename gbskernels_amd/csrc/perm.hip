// perm.hip -- launches of the Glynn permanent kernels (perm_impl.hpp): the split
// table, one size per launch, and the multi-size launch of a batch's buckets.
#include <algorithm>

#include "launch_split.hpp"
#include "perm_impl.hpp"
#include "perm_mix.hpp"
#include "perm_tune.hpp"

namespace gbsk {

// ------------------------------------------------------------- split table
// Read with relaxed atomics by every launch; written only by the tuning entry
// point (documented: not while evaluations are in flight).
static int g_lane_log2[2][PERM_MAX_N + 1];
[[maybe_unused]] static const bool g_lane_log2_init = [] {
  for (int f = 0; f < 2; ++f)
    for (int n = 0; n <= PERM_MAX_N; ++n) g_lane_log2[f][n] = kPermLaneLog2[f][n];
  return true;
}();

template <int N, int DD>
static PermSplit split_of() {
  using C = PermCfg<N, DD>;
  const int t = __atomic_load_n(&g_lane_log2[DD][N], __ATOMIC_RELAXED);
  const int M = t < C::MLIM ? t : C::MLIM;
  return PermSplit{M, 1 << (C::MLIM - M)};
}

static size_t perm_chunk_bytes(int mode) { return mode == PERM_DDCERT ? 16 + 16 + 8 : 16 + 16; }

template <int N, int MODE>
static int launch_perm_n(const cplx* d_in, int B, cplx* d_out, double* d_aux, void* ws, size_t ws_size,
                         hipStream_t st) {
  using C = PermCfg<N, perm_is_dd(MODE) ? 1 : 0>;
  constexpr int MPW = 64 / C::LPM;
  // the split is read once: the workspace check and the launches agree
  const PermSplit sp = split_of<N, perm_is_dd(MODE) ? 1 : 0>();
  const int M = sp.M, W = sp.W;
  if (W > 1 && ws_size < (size_t)B * W * perm_chunk_bytes(MODE)) return GBSK_ERR_WORKSPACE;
  // batches above the launch limit run as consecutive sub-batches (same stream,
  // the workspace reused), matrices of a sub-batch a multiple of 8 groups so the
  // XCD mapping is unchanged
  const int64_t max_b = launch_rows(W, 8) * MPW;
  for (int64_t b0 = 0; b0 < B; b0 += max_b) {
    const int Bs = (int)((B - b0) < max_b ? (B - b0) : max_b);
    const cplx* in = d_in + b0 * N * N;
    cplx* out = d_out + b0;
    double* aux = d_aux ? d_aux + b0 : nullptr;
    const int64_t groups = ((int64_t)Bs + MPW - 1) / MPW;
    const int g8 = groups < 8 ? (int)groups : 8;
    const int64_t grid = perm_grid(groups, W);
    if (W == 1) {
      hipLaunchKernelGGL((perm_kernel<N, MODE>), dim3((unsigned)grid), dim3(64), 0, st, in, Bs, out, aux, g8, M, W);
    } else {
      // partials: values [Bs][W] cplx, then [Bs][W] of 16 bytes (kappa / bound
      // doubles, or the dd low parts), then (certified dd) [Bs][W] bounds
      cplx* part = reinterpret_cast<cplx*>(ws);
      double* part_aux = reinterpret_cast<double*>(part + (size_t)Bs * W);
      hipLaunchKernelGGL((perm_kernel<N, MODE>), dim3((unsigned)grid), dim3(64), 0, st, in, Bs, part, part_aux, g8,
                         M, W);
      hipLaunchKernelGGL((perm_reduce_kernel<N, MODE>), dim3((unsigned)((Bs + 255) / 256)), dim3(256), 0, st, part,
                         part_aux, Bs, out, aux, M, W);
    }
  }
  return (int)hipGetLastError();
}

// n == 0: perm = 1 (empty product); kappa indicator 1, certificate 0 (exact)
__global__ void perm_n0_kernel(int B, cplx* out, double* aux, double auxval) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B) return;
  out[b] = cplx{1.0, 0.0};
  if (aux) aux[b] = auxval;
}



template <int MODE, int... Ns>
static int dispatch_perm(int n, const cplx* d_in, int B, cplx* d_out, double* d_aux, void* ws, size_t ws_size,
                         hipStream_t st, std::integer_sequence<int, Ns...>) {
  int rc = GBSK_ERR_DIM;
  ((n == Ns ? (rc = launch_perm_n<Ns, MODE>(d_in, B, d_out, d_aux, ws, ws_size, st), 0) : 0), ...);
  return rc;
}

template <int... Ns>
static PermSplit split_dispatch(int n, int family, std::integer_sequence<int, Ns...>) {
  PermSplit r{0, 1};
  ((n == Ns ? (r = family ? split_of<Ns, 1>() : split_of<Ns, 0>(), 0) : 0), ...);
  return r;
}

template <int... Ns>
static int mpw_dispatch(int n, std::integer_sequence<int, Ns...>) {
  int r = 1;
  ((n == Ns ? (r = 64 / PermCfg<Ns, 0>::LPM, 0) : 0), ...);
  return r;
}
static int perm_mpw(int n) { return mpw_dispatch(n, PermSizes{}); }
template <int... Ns>
static bool mixed_dispatch(int n, std::integer_sequence<int, Ns...>) {
  return ((n == Ns && perm_mixed<Ns>()) || ...);
}

PermSplit perm_split(int n, int family) {
  if (n < 1 || n > PERM_MAX_N) return PermSplit{0, 1};
  return split_dispatch(n, family ? 1 : 0, PermSizes{});
}

int perm_lane_log2_get(int family, int n) {
  if ((family != 0 && family != 1) || n < 0 || n > PERM_MAX_N) return GBSK_ERR_ARG;
  return __atomic_load_n(&g_lane_log2[family][n], __ATOMIC_RELAXED);
}

// at least 2^LOGMIN terms per lane (16 fp64, 4 dd: the per-lane start costs n^2
// updates) and at most 2^27 (every n <= 28 then runs one workgroup per matrix)
int perm_lane_log2_set(int family, int n, int log2_terms) {
  if ((family != 0 && family != 1) || n < 0 || n > PERM_MAX_N) return GBSK_ERR_ARG;
  if (log2_terms < (family ? 2 : 4) || log2_terms > 27) return GBSK_ERR_ARG;
  __atomic_store_n(&g_lane_log2[family][n], log2_terms, __ATOMIC_RELAXED);
  return 0;
}

size_t perm_workspace_bytes(int n, int mode, int B) {
  if (n < 1 || n > PERM_MAX_N || B <= 0) return 0;
  const PermSplit sp = perm_split(n, perm_is_dd(mode) ? 1 : 0);
  return sp.W > 1 ? (size_t)B * sp.W * perm_chunk_bytes(mode) : 0;
}

int perm_launch(int n, int mode, const cplx* d_in, int B, cplx* d_out, double* d_aux, void* ws, size_t ws_size,
                hipStream_t st) {
  if (B <= 0) return 0;
  if (n < 0 || n > PERM_MAX_N) return GBSK_ERR_DIM;
  if (n == 0) {
    hipLaunchKernelGGL(perm_n0_kernel, dim3((B + 255) / 256), dim3(256), 0, st, B, d_out,
                       (mode == PERM_KAPPA || mode == PERM_CERT || mode == PERM_DDCERT) ? d_aux : nullptr,
                       mode == PERM_KAPPA ? 1.0 : 0.0);
    return (int)hipGetLastError();
  }
  switch (mode) {
    case PERM_FP64: return dispatch_perm<PERM_FP64>(n, d_in, B, d_out, d_aux, ws, ws_size, st, PermSizes{});
    case PERM_KAPPA: return dispatch_perm<PERM_KAPPA>(n, d_in, B, d_out, d_aux, ws, ws_size, st, PermSizes{});
    case PERM_DD: return dispatch_perm<PERM_DD>(n, d_in, B, d_out, d_aux, ws, ws_size, st, PermSizes{});
    case PERM_CERT: return dispatch_perm<PERM_CERT>(n, d_in, B, d_out, d_aux, ws, ws_size, st, PermSizes{});
    case PERM_DDCERT: return dispatch_perm<PERM_DDCERT>(n, d_in, B, d_out, d_aux, ws, ws_size, st, PermSizes{});
  }
  return GBSK_ERR_ARG;
}

int perm_launch_multi(int mode, const PermJob* jobs, int njobs, hipStream_t st) {
  if (njobs < 0 || njobs > PERM_MAX_JOBS || (njobs && !jobs)) return GBSK_ERR_ARG;
  const bool mix = mode == PERM_FP64 || mode == PERM_KAPPA;
  PermMix m;
  m.count = 0;
  int64_t wgs = 0, reds = 0;
  bool big = true;
  auto flush = [&]() {
    if (!m.count) return;
    m.wg_begin[m.count] = (unsigned)wgs;
    m.red_begin[m.count] = (unsigned)reds;
    if (mode == PERM_KAPPA)
      big ? perm_mix_launch<PERM_KAPPA, true>(m, st) : perm_mix_launch<PERM_KAPPA, false>(m, st);
    else
      big ? perm_mix_launch<PERM_FP64, true>(m, st) : perm_mix_launch<PERM_FP64, false>(m, st);
    m.count = 0;
    wgs = reds = 0;
  };
  // largest sides first: their workgroups run longest
  int order[PERM_MAX_JOBS];
  for (int i = 0; i < njobs; ++i) order[i] = i;
  std::stable_sort(order, order + njobs, [&](int x, int y) { return jobs[x].n > jobs[y].n; });
  for (int k = 0; k < njobs; ++k) {
    const PermJob& j = jobs[order[k]];
    if (j.B <= 0) continue;
    if (j.n < 0 || j.n > PERM_MAX_N) return GBSK_ERR_DIM;
    const PermSplit sp = perm_split(j.n, 0);
    const int mpw = perm_mpw(j.n);
    const int64_t groups = ((int64_t)j.B + mpw - 1) / mpw;
    const int g8 = groups < 8 ? (int)groups : 8;
    const int64_t grid = perm_grid(groups, sp.W);
    if (!mix || !mixed_dispatch(j.n, PermSizes{}) || grid > LAUNCH_WAVES) {
      const int rc = perm_launch(j.n, mode, j.in, j.B, j.out, j.aux, j.ws, j.ws_size, st);
      if (rc) return rc;
      continue;
    }
    if (sp.W > 1 && j.ws_size < (size_t)j.B * sp.W * perm_chunk_bytes(mode)) return GBSK_ERR_WORKSPACE;
    const bool side = j.n >= PERM_MIX_BIG;  // sorted by side: changes once
    if (side != big || wgs + grid > LAUNCH_WAVES) flush();
    big = side;
    const int q = m.count++;
    cplx* part = reinterpret_cast<cplx*>(j.ws);
    m.in[q] = j.in;
    m.out[q] = j.out;
    m.aux[q] = j.aux;
    m.part[q] = part;
    m.part_aux[q] = sp.W > 1 ? reinterpret_cast<double*>(part + (size_t)j.B * sp.W) : nullptr;
    m.n[q] = (uint8_t)j.n;
    m.g8[q] = (uint8_t)g8;
    m.M[q] = (uint8_t)sp.M;
    m.W[q] = sp.W;
    m.B[q] = j.B;
    m.wg_begin[q] = (unsigned)wgs;
    m.red_begin[q] = (unsigned)reds;
    wgs += grid;
    if (sp.W > 1) reds += ((int64_t)j.B + 63) / 64;
  }
  flush();
  return (int)hipGetLastError();
}

}  // namespace gbsk
