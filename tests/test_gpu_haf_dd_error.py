"""Error of the double-double hafnians of sides 14 .. 20 at their own level, 2^-106 of
sum |term|. Two entries of each matrix are solved for so that the value cancels to
that level and the double that comes back still resolves it; quad values are
exact to 2^-113."""
import sys
from pathlib import Path

import numpy as np
import pytest

from conftest import rng_symmetric

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "gbskernels_amd" / "ext"))
pytestmark = pytest.mark.gpu

# (function, side, matrices, rms error of the power-trace kernels on 512 / 256 / 96 / 48
# such matrices). The root mean square of n errors of kurtosis up to 6 has standard
# deviation sqrt(5 / 4n) of itself: three of those are allowed for.
CASES = [("haf", 14, 192, 0.216), ("haf", 16, 96, 0.183), ("haf", 18, 32, 0.160), ("haf", 20, 16, 0.149),
         ("lhaf", 14, 192, 0.255), ("lhaf", 16, 96, 0.196), ("lhaf", 18, 32, 0.170), ("lhaf", 20, 16, 0.147)]


def cancelling(oracle, func, N, B, seed):
    """B symmetric matrices whose value is about 2^-113 of sum |term|, the values
    in quad and sum |term|. The value is linear in each entry: the first takes it
    to 2^-53, the second, small, the rest of the way."""
    f = getattr(oracle, func + "_q")
    A = rng_symmetric(B, N, seed, 0.5 / N ** 0.5)
    rows = np.stack([np.random.default_rng(seed + 1 + b).permutation(N)[:4] for b in range(B)])

    def put(q, v):
        for b, x in enumerate(rows):
            A[b, x[q], x[q + 1]] = A[b, x[q + 1], x[q]] = v[b]

    def minors(q):
        return f(np.stack([np.delete(np.delete(A[b], x[q:q + 2], 0), x[q:q + 2], 1) for b, x in enumerate(rows)]))

    put(0, np.zeros(B))
    put(2, np.zeros(B))
    put(0, -f(A) / minors(0))
    put(2, -f(A) / minors(2))
    return A, f(A), getattr(oracle, func + "_abs")(A)


@pytest.mark.parametrize("func,N,B,power_trace", CASES)
def test_dd_error_no_larger_than_the_power_trace(oracle, func, N, B, power_trace):
    import gbskernels_ext as ext
    print(f"{func} dd error N={N}", flush=True)
    A, want, scale = cancelling(oracle, func, N, B, 7000 + N)
    got = getattr(ext, func + "_dd")(A)
    cert, bound = getattr(ext, func + "_dd_certified")(A)
    err = np.abs(got - want) / scale * 2.0 ** 106
    assert np.sqrt(np.mean(err ** 2)) <= power_trace * (1 + 3 * np.sqrt(5 / (4 * B)))
    assert np.array_equal(cert, got)
    assert np.all(np.abs(got - want) <= bound + 2.0 ** -113 * scale)
