"""Width of the certified bounds of sides 14 .. 20, relative to sum |term|, against
the power-trace kernels' on the same kind of matrices (complex, symmetric,
Gaussian): no wider in fp64, at most 2.5 times in double-double."""
import sys
from pathlib import Path

import numpy as np
import pytest

from conftest import rng_symmetric
from test_gpu_haf_dd_error import cancelling

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "gbskernels_amd" / "ext"))
pytestmark = pytest.mark.gpu

# medians of the power trace's bounds: fp64 in 2^-53 sum |term|, dd in 2^-106
FP64 = {"haf": {14: 3588, 16: 6860, 18: 20454, 20: 42970}, "lhaf": {14: 6093, 16: 14928, 18: 31377, 20: 74030}}
DD = {"haf": {14: 519, 16: 984, 18: 2069}, "lhaf": {14: 930, 16: 1962, 18: 3792}}


@pytest.mark.parametrize("N", [14, 16, 18, 20])
@pytest.mark.parametrize("func", ["haf", "lhaf"])
def test_fp64_bounds_no_wider_than_the_power_trace(func, N):
    import gbskernels_ext as ext
    print(f"{func} certified width N={N}", flush=True)
    A = rng_symmetric(96, N, 5100 + N, 0.5)
    bound = getattr(ext, func + "_certified")(A)[1]
    scale = getattr(ext, func + "_kappa")(A)[1]
    assert np.median(bound / scale) * 2.0 ** 53 <= FP64[func][N]


@pytest.mark.parametrize("N", [14, 16, 18])
@pytest.mark.parametrize("func", ["haf", "lhaf"])
def test_dd_bounds_within_reach_of_the_power_trace(oracle, func, N):
    import gbskernels_ext as ext
    print(f"{func} dd certified width N={N}", flush=True)
    A, _, scale = cancelling(oracle, func, N, 48, 5200 + N)
    bound = getattr(ext, func + "_dd_certified")(A)[1]
    assert np.median(bound / scale) * 2.0 ** 106 <= 2.5 * DD[func][N]
