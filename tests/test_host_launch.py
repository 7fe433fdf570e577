"""Host arithmetic of the launches (no GPU): workspace sizes, and how batches are
cut so that every launch stays below HIP's 2^32 work-items."""
import ctypes
import subprocess
from pathlib import Path

import pytest

from gbskernels_amd import _lib

LIMIT = 2 ** 26  # waves of 64 work-items: 2^32


@pytest.mark.parametrize("N", range(14, 30, 2))
@pytest.mark.parametrize("func", ["haf", "lhaf"])
def test_tree_workspace_is_what_the_kernels_write(func, N):
    """One partial (value and double) per include pattern of all but four pairs."""
    for tier, elem in (("fp64", 16), ("kappa", 16), ("certified", 16), ("dd", 32), ("dd_certified", 32)):
        got = _lib.lib().gbs_workspace_bytes(_lib.FUNCS[func], _lib.TIERS[tier], N, 1000)
        assert got == 1000 * 2 ** (N // 2 - 4) * (elem + 8)


# The split header is plain C++: the test compiles it and prints, for each side,
# the waves of one instance and how buckets around the limit are cut.
SPLIT = r"""
#include <cstdio>
#include <initializer_list>
#include "haf_parts.hpp"
#include "launch_split.hpp"
using namespace gbsk;
int main() {
  for (int N = 2; N <= TREE_MAX_N; N += 2) {
    const long long w = haf_launch_waves(N), most = launch_rows(w);
    for (long long B : {1ll, most - 1, most, most + 1, 3 * most, 3 * most + 5, 2147483647ll})
      for (int first : {0, 1, 700}) {  // waves an earlier bucket holds
        LaunchRoom room;
        room.take(first, 1);
        std::printf("haf %d %lld %lld %d", N, w, B, first);
        for (long long b0 = 0; b0 < B;) {
          const long long n = room.take(B - b0, w);
          if (n == 0) { std::printf(" |"); room = LaunchRoom{}; continue; }
          std::printf(" %lld", n);
          b0 += n;
        }
        std::printf("\n");
      }
  }
}
"""


def run_split(tmp_path, code):
    src, exe = tmp_path / "split.cpp", tmp_path / "split"
    src.write_text(code)
    csrc = Path(_lib.__file__).parent / "csrc"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{csrc}", str(src), "-o", str(exe)], check=True)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines()


def test_hafnian_buckets_stay_below_the_launch_limit(tmp_path):
    waves = {}
    for line in run_split(tmp_path, SPLIT):
        _, N, w, B, first, *cut = line.split()
        N, w, B, used = int(N), int(w), int(B), int(first)
        waves[N] = w
        taken = 0
        for c in cut:
            if c == "|":
                assert used + w > LIMIT - 4 or used == 0, line  # cut only where the next row does not fit
                assert used > 0
                used = 0
            else:
                used += int(c) * w
                taken += int(c)
                # 64 lanes a wave, and a reduction of four waves a workgroup over as many instances
                assert 0 < used and 64 * used < 2 ** 32 and (used + 3) // 4 * 256 < 2 ** 32, line
        assert taken == B, line
    assert all(waves[N] == 2 ** (N // 2 - 4) for N in range(14, 30, 2))
    assert waves[12] == 2 and waves[2] == 1


PERM = r"""
#include <cstdio>
#include <initializer_list>
#include "launch_split.hpp"
using namespace gbsk;
int main() {
  for (int lw = 0; lw <= 19; ++lw) {  // workgroups a matrix: 1 .. 2^19 (two terms a lane)
    const int W = 1 << lw;
    const long long most = launch_rows(W, 8);
    for (long long g : {most - 1, most, most + 1})
      std::printf("%d %lld %lld %lld\n", W, most, g, (long long)perm_grid(g, W));
  }
}
"""


def test_permanent_sub_batches_stay_below_the_launch_limit(tmp_path):
    for line in run_split(tmp_path, PERM):
        W, most, groups, grid = map(int, line.split())
        assert most >= 8 and most % 8 == 0 and groups * W <= grid <= (groups + 7) * W
        if groups <= most:
            assert grid * 64 < 2 ** 32, line
    # what the split gives for every size and chunking that can be set
    k, w = ctypes.c_int(), ctypes.c_int()
    L = _lib.lib()
    for family in (0, 1):
        for n in range(1, 29):
            keep = ctypes.c_int()
            assert L.gbs_perm_get_lane_log2(family, n, ctypes.byref(keep)) == 0
            try:
                assert L.gbs_perm_set_lane_log2(family, n, 2 if family else 4) == 0
                assert L.gbs_perm_split(family, n, ctypes.byref(k), ctypes.byref(w)) == 0
                assert w.value <= 2 ** 19
            finally:
                assert L.gbs_perm_set_lane_log2(family, n, keep.value) == 0


ROWS = r"""
#include <cstdio>
#include "launch_split.hpp"
int main() {
  for (int t1 = 0; t1 <= 21; ++t1)  // workgroups an instance of the torontonian: 2^t1
    std::printf("%d %lld\n", 1 << t1, (long long)gbsk::launch_rows((int64_t)1 << t1));
  std::printf("4 %lld\n", (long long)gbsk::LAUNCH_WAVES / 4);  // four patterns of the sieve a workgroup
}
"""


def test_rows_of_one_launch(tmp_path):
    for line in run_split(tmp_path, ROWS):
        waves, rows = map(int, line.split())
        assert rows >= 1 and rows * waves * 64 < 2 ** 32 and ((rows + 3) // 4 * 256 < 2 ** 32)
