"""Double-double permanents split every row on its own grid (high parts summed
exactly, low parts apart): values against exact rational permanents on rows the
split could go wrong on. The tolerance is the certified bound, which the same
kernel derives; the plain tier must return the same bits."""
import itertools
import sys
from fractions import Fraction
from pathlib import Path

import numpy as np
import pytest

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "gbskernels_amd" / "ext"))
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ext():
    import gbskernels_ext
    return gbskernels_ext


def exact_perm(A):
    """Permanent in rationals by subsets of columns, row by row."""
    n = A.shape[0]
    re = [[Fraction(float(A[r, c].real)) for c in range(n)] for r in range(n)]
    im = [[Fraction(float(A[r, c].imag)) for c in range(n)] for r in range(n)]
    P = {0: (Fraction(1), Fraction(0))}
    for r in range(n):
        Q = {}
        for S in itertools.combinations(range(n), r + 1):
            key, x, y = sum(1 << c for c in S), Fraction(0), Fraction(0)
            for c in S:
                a, b = P[key ^ (1 << c)]
                x += a * re[r][c] - b * im[r][c]
                y += a * im[r][c] + b * re[r][c]
            Q[key] = (x, y)
        P = Q
    return P[(1 << n) - 1]


def stacks(kind, n, rng):
    A = rng.standard_normal((3, n, n)) + 1j * rng.standard_normal((3, n, n))
    if kind == "row scales":
        A *= np.exp2(rng.integers(-90, 90, (3, n, 1)))
    elif kind == "entry scales":
        A *= np.exp2(rng.integers(-70, 70, (3, n, n)))
    elif kind == "zero and real rows":
        A[0, n - 1] = 0.0
        A[1].imag[0] = 0.0
        A[2].real[n - 1] = 0.0
    elif kind == "powers of two":
        A = np.exp2(rng.integers(-40, 40, (3, n, n))) * (1 - 1j)
    return np.ascontiguousarray(A)


@pytest.mark.parametrize("kind", ["plain", "row scales", "entry scales", "zero and real rows", "powers of two"])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 8, 9])
def test_perm_dd_split_rows(ext, kind, n):
    print(f"perm dd split rows n={n} {kind}", flush=True)
    A = stacks(kind, n, np.random.default_rng(4000 + n))
    v, b = ext.perm_dd_certified(A)
    assert np.array_equal(v, ext.perm_dd(A))
    assert np.all(np.isfinite(b))
    for k in range(3):
        x, y = exact_perm(A[k])
        off = abs(Fraction(float(v[k].real)) - x) + abs(Fraction(float(v[k].imag)) - y)
        assert off <= Fraction(float(b[k]))


@pytest.mark.parametrize("n", [2, 7, 12])
def test_perm_dd_non_finite_rows(ext, n):
    """One infinite or NaN entry reaches its own matrix's value only."""
    rng = np.random.default_rng(4100 + n)
    A = rng.standard_normal((4, n, n)) + 1j * rng.standard_normal((4, n, n))
    good = ext.perm_dd(A)
    A[1, n - 1, 0] = np.inf
    A[2, 0, n - 1] = np.nan
    v = ext.perm_dd(A)
    assert not np.isfinite(v[1]) and not np.isfinite(v[2])
    assert np.array_equal(v[[0, 3]], good[[0, 3]])
