// perm_mix.hpp -- permanents of several sizes in one launch (fp64 and kappa): the
// buckets of a mixed batch. A bucket of a few matrices is a few waves that each
// walk 2^9 terms (75-470 us from n = 15 to 24 on MI355X) on an otherwise empty
// device, and the sizes ran one after another on a stream. Here every size's
// workgroups are in one grid, largest sides first, and each runs its size's own
// code (perm_workgroup, same split: values are the same bits). Measured, window
// of 2048 requests up to side 24 (kappa): the batch's device time 2230 -> 1050 us.
#pragma once

#include "perm.hpp"

namespace gbsk {

// Sizes one launch carries: those whose matrices fit the LDS that lets two waves
// a SIMD run (20 KB a workgroup; all but n = 5, 64 matrices of which take 25 KB).
constexpr int PERM_MIX_LDS = 1280;  // complex numbers
template <int N>
constexpr bool perm_mixed() { return (64 / PermCfg<N, 0>::LPM) * N * N <= PERM_MIX_LDS; }
// Two kernels: sides from PERM_MIX_BIG on fill 256 VGPRs and spill a few, and a
// kernel with scratch makes its queue allocate it at its first launch (a first
// batch of small sides 820 -> 1170 us), so the smaller sides have one of their own.
constexpr int PERM_MIX_BIG = 14;

struct PermMix {  // by value in the kernel argument block
  const cplx* in[PERM_MAX_JOBS];
  cplx* out[PERM_MAX_JOBS];
  double* aux[PERM_MAX_JOBS];
  cplx* part[PERM_MAX_JOBS];        // chunk partials (W > 1), then part_aux
  double* part_aux[PERM_MAX_JOBS];
  int B[PERM_MAX_JOBS], W[PERM_MAX_JOBS];
  uint8_t n[PERM_MAX_JOBS], g8[PERM_MAX_JOBS], M[PERM_MAX_JOBS];
  unsigned wg_begin[PERM_MAX_JOBS + 1];   // first workgroup of each bucket
  unsigned red_begin[PERM_MAX_JOBS + 1];  // the same of the chunk reduction, 64 matrices a workgroup
  int count;
};

template <int MODE, bool BIG>
void perm_mix_launch(const PermMix& m, hipStream_t st);

}  // namespace gbsk
