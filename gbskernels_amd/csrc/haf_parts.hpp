// haf_parts.hpp -- partials per instance of the hafnian kernels: plain arithmetic, the
// same on the host (workspace sizes, launch splits) and in the kernels.
#pragma once

namespace gbsk {

// Sides 14..28 run the series tree (haf_tree.hpp): one partial per include pattern
// of the leading pairs, all but TREE_T2. Smaller sides run the power-trace kernels.
constexpr int TREE_MIN_N = 14;
constexpr int TREE_MAX_N = 28;
// Pairs left to the tree of one workgroup (one wave); the h - 4 leading pairs'
// include / exclude patterns are separate workgroups. A level's series tasks
// then take up to 40 lanes (60 with the loop row) at two lanes a task, and the
// series of a workgroup (18.9 KB at N = 24, 12.1 KB at N = 16) leave room for 8 and
// 12 waves a CU. Five pairs with one lane a task took 54 KB at N = 24, two waves
// a CU: 3.37 ms where this takes 1.40.
constexpr int TREE_T2 = 4;
constexpr int HAF_PHASE_MAX_N = TREE_MIN_N - 2;
constexpr int tree_parts(int N) { return 1 << (N / 2 - TREE_T2); }

// Work split of a power-trace phase: its C(n, m) subsets are cut into chunks of
// HAF_CHUNK_ITERS * G consecutive subsets (G = 64 / S per wave iteration), one
// workgroup per (instance, chunk), so that large N runs many waves per instance.
// The split depends on (N, S) only; chunk partials are summed in chunk order.
constexpr int HAF_CHUNK_ITERS = 1;
constexpr int haf_chunk_size(int S) { return HAF_CHUNK_ITERS * (64 / S); }
constexpr int haf_binom(int n, int k) {
  if (k < 0 || k > n) return 0;
  int r = 1;
  for (int i = 1; i <= k; ++i) r = r * (n - k + i) / i;
  return r;
}
constexpr int haf_nchunks(int n, int S) {
  const int c = haf_binom(n, S / 2), ch = haf_chunk_size(S);
  return (c + ch - 1) / ch;
}
// partial slots per instance (all phases) and the first slot of phase S
constexpr int haf_nparts(int n) {
  int t = 0;
  for (int m = 1; m <= n; ++m) t += haf_nchunks(n, 2 * m);
  return t;
}
constexpr int haf_part_offset(int n, int S) {
  int t = 0;
  for (int m = 1; m < S / 2; ++m) t += haf_nchunks(n, 2 * m);
  return t;
}

// partials of one instance of side N (even, 2 .. TREE_MAX_N)
constexpr int haf_parts(int N) { return N > HAF_PHASE_MAX_N ? tree_parts(N) : haf_nparts(N / 2); }

// waves one instance adds to the largest of its launches (at least one: the reduction's)
constexpr int haf_launch_waves(int N) {
  if (N > HAF_PHASE_MAX_N) return tree_parts(N);
  int most = 1;
  for (int S = 2; S <= N; S += 2) most = haf_nchunks(N / 2, S) > most ? haf_nchunks(N / 2, S) : most;
  return most;
}

}  // namespace gbsk
