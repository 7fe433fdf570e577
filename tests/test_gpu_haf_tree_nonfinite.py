"""Sides 14..28: a NaN or an infinity in one place of one triangle, wherever it is,
makes the value NaN and the certificate infinite, in that instance only."""
import sys
from pathlib import Path

import numpy as np
import pytest

from conftest import rng_symmetric

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "gbskernels_amd" / "ext"))
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tier", ["", "_kappa", "_certified", "_dd", "_dd_certified"])
@pytest.mark.parametrize("func", ["haf", "lhaf"])
@pytest.mark.parametrize("N", [14, 20, 28])
def test_one_entry_of_one_triangle(func, tier, N):
    import gbskernels_ext as ext
    print(f"{func}{tier} N={N}", flush=True)
    f = getattr(ext, func + tier)
    # leading block, trailing block (the last eight rows) and between them
    places = [(5, 2), (2, 5), (N - 1, N - 3), (N - 3, N - 1), (N - 1, 0), (0, N - 1), (N - 7, N - 8), (N - 8, N - 7)]
    if N == 28:
        places = places[2:5]
    A = rng_symmetric(2 * len(places), N, 14000 + N, 0.3)
    want = f(A)
    B = A.copy()
    for k, p in enumerate(places):
        B[2 * k][p] = (np.nan, np.inf, complex(0, -np.inf))[k % 3]
    got = f(B)
    want, got = [r if isinstance(r, tuple) else (r,) for r in (want, got)]
    for w, g in zip(want, got):
        assert np.array_equal(g[1::2], w[1::2])
        assert not np.any(np.isfinite(g[::2]))
