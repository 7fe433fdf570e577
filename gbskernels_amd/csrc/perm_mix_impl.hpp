// perm_mix_impl.hpp -- kernels of perm_mix.hpp, one tier per translation unit.
#pragma once

#include "perm_impl.hpp"
#include "perm_mix.hpp"

namespace gbsk {

// runs N's workgroup if the launch carries that size
template <int N, int MODE, bool BIG>
__device__ __forceinline__ void perm_mix_one(const PermMix& m, int q, cplx* out, double* aux, int64_t wg, cplx* lds) {
  if constexpr (perm_mixed<N>() && (N >= PERM_MIX_BIG) == BIG)
    perm_workgroup<N, MODE>(m.in[q], m.B[q], out, aux, m.g8[q], m.M[q], m.W[q], wg, lds);
}

template <int MODE, bool BIG, int... Ns>
__device__ __forceinline__ void perm_mix_run(const PermMix& m, int q, int64_t wg, cplx* lds,
                                             std::integer_sequence<int, Ns...>) {
  const int n = m.n[q], W = m.W[q];
  cplx* const out = W > 1 ? m.part[q] : m.out[q];
  double* const aux = W > 1 ? m.part_aux[q] : m.aux[q];
  ((n == Ns ? (perm_mix_one<Ns, MODE, BIG>(m, q, out, aux, wg, lds), 0) : 0), ...);
}

template <int MODE, bool BIG>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(perm_min_waves<MODE>()))) void perm_mix_kernel(
    const PermMix m) {
  __shared__ cplx lds[PERM_MIX_LDS];
  int q = 0;  // this workgroup's bucket
  while (q + 1 < m.count && blockIdx.x >= m.wg_begin[q + 1]) ++q;
  perm_mix_run<MODE, BIG>(m, q, (int64_t)blockIdx.x - m.wg_begin[q], lds, PermSizes{});
}

template <int MODE, int... Ns>
__device__ __forceinline__ void perm_mix_reduce_run(int n, const cplx* part, const double* part_aux, int B, cplx* out,
                                                    double* aux, int M, int W, int64_t b,
                                                    std::integer_sequence<int, Ns...>) {
  ((n == Ns ? (perm_reduce<Ns, MODE>(part, part_aux, B, out, aux, M, W, b), 0) : 0), ...);
}

template <int MODE>
__global__ __launch_bounds__(64) void perm_mix_reduce_kernel(const PermMix m) {
  int q = 0;
  while (q + 1 < m.count && blockIdx.x >= m.red_begin[q + 1]) ++q;
  perm_mix_reduce_run<MODE>(m.n[q], m.part[q], m.part_aux[q], m.B[q], m.out[q], m.aux[q], m.M[q], m.W[q],
                            (int64_t)(blockIdx.x - m.red_begin[q]) * 64 + threadIdx.x, PermSizes{});
}

template <int MODE, bool BIG>
void perm_mix_launch(const PermMix& m, hipStream_t st) {
  hipLaunchKernelGGL((perm_mix_kernel<MODE, BIG>), dim3(m.wg_begin[m.count]), dim3(64), 0, st, m);
  if (m.red_begin[m.count])
    hipLaunchKernelGGL((perm_mix_reduce_kernel<MODE>), dim3(m.red_begin[m.count]), dim3(64), 0, st, m);
}

}  // namespace gbsk
