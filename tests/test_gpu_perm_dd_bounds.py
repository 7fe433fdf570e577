"""Width of the certified double-double permanents' bounds where the value cancels, so
that the bound shows: the last row the negative of the first and one column 1e-9
times the others. No wider, relative to sum |term|, than with double-double
additions of the row sums; with rows that span 24 decades at most 2.5 times."""
import sys
from pathlib import Path

import numpy as np
import pytest

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "gbskernels_amd" / "ext"))
pytestmark = pytest.mark.gpu

# medians of bound / sum |term| in 2^-106 with double-double additions, these inputs
CANCELLING = {4: 2.76e6, 8: 5.79e5, 12: 1.22e5, 14: 7.13e4, 16: 3.70e4}
WILD = {6: 7.12e9, 8: 3.41e8, 10: 1.06e8}


def draw(n):
    rng = np.random.default_rng(n)
    B = 700 if n < 12 else 40
    A = rng.standard_normal((B, n, n)) + 1j * rng.standard_normal((B, n, n))
    wild = A * 10.0 ** rng.integers(-12, 13, A.shape)
    A[:, -1] = -A[:, 0]
    A[:, :, -1] *= 1e-9
    return A, wild


def median(oracle, A):
    import gbskernels_ext as ext
    return np.median(ext.perm_dd_certified(A)[1] / oracle.perm_abs(A)) * 2.0 ** 106


@pytest.mark.parametrize("n", CANCELLING)
def test_cancelling(oracle, n):
    print(f"perm dd bound n={n}", flush=True)
    assert median(oracle, draw(n)[0]) <= 1.01 * CANCELLING[n]  # the constants have three digits


@pytest.mark.parametrize("n", WILD)
def test_rows_of_many_scales(oracle, n):
    print(f"perm dd bound, wild rows n={n}", flush=True)
    A = draw(n)[1]
    assert median(oracle, A) <= 2.5 * WILD[n]


@pytest.mark.parametrize("n", [3, 4, 5, 9])
@pytest.mark.parametrize("spread", [45, 48, 49, 50, 51, 53, 60, 110])
def test_values_enclosed_around_the_line(oracle, n, spread):
    """Rows whose smallest entry lies `spread` binary orders below the largest: on both
    sides of the line from which low sums may round."""
    import gbskernels_ext as ext
    print(f"perm dd line n={n} spread={spread}", flush=True)
    rng = np.random.default_rng(100 * n + spread)
    A = rng.standard_normal((200, n, n)) + 1j * rng.standard_normal((200, n, n))
    A[:, :, rng.integers(n)] *= 2.0 ** -spread
    A[:, -1] = -A[:, 0] * (1 + 2.0 ** -30)
    v, b = ext.perm_dd_certified(A)
    assert np.array_equal(v, ext.perm_dd(A))
    q = oracle.perm_q(A)
    assert np.all(np.abs(v - q) <= b + 2.0 ** -52 * np.abs(q) * 2.0 ** -50 + 2.0 ** -112 * oracle.perm_abs(A))
