"""The series-tree hafnian kernels (sides 14..28) at every side and tier: values
against the oracle or against products of smaller hafnians, kappa sums against
the oracle's, certified values bit-identical to the plain tiers' and enclosing,
and values independent of the batch around them. Tolerances are multiples of
the summation's own scale, 256 N eps sum |term| (the power-trace tests' bound)."""
import math
import sys
from pathlib import Path

import numpy as np
import pytest

from conftest import rel_err, rng_symmetric

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "gbskernels_amd" / "ext"))
pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52
SIDES = [14, 16, 18, 20, 22, 24, 26, 28]


@pytest.fixture(scope="module")
def ext():
    import gbskernels_ext
    return gbskernels_ext


def scattered_blocks(N, seed):
    """Two independent symmetric blocks (12 and N - 12 rows) under one random
    row order, which the index pairs do not respect: (matrix, the two blocks)."""
    g = np.random.default_rng(seed)
    P, Q = rng_symmetric(1, 12, seed + 1, 0.5)[0], rng_symmetric(1, N - 12, seed + 2, 0.5)[0]
    order = g.permutation(N)
    A = np.zeros((N, N), complex)
    A[np.ix_(order[:12], order[:12])] = P
    A[np.ix_(order[12:], order[12:])] = Q
    return A, P, Q


@pytest.mark.parametrize("N", SIDES)
@pytest.mark.parametrize("func", ["haf", "lhaf"])
def test_every_tier_on_block_products(ext, oracle, func, N):
    print(f"{func} tree N={N}", flush=True)
    A, P, Q = scattered_blocks(N, 40 * N)
    f = getattr(oracle, f"{func}_q")
    want = f(P[None])[0] * f(Q[None])[0]
    v = getattr(ext, func)(A[None])
    k, a = getattr(ext, f"{func}_kappa")(A[None])
    c, cb = getattr(ext, f"{func}_certified")(A[None])
    d = getattr(ext, f"{func}_dd")(A[None])
    e, eb = getattr(ext, f"{func}_dd_certified")(A[None])
    assert np.array_equal(v, k) and np.array_equal(v, c) and np.array_equal(d, e)
    assert abs(v[0] - want) <= 256.0 * N * EPS * a[0]
    slack = 4 * EPS * abs(want)  # the product of two oracle values, rounded
    assert abs(d[0] - want) <= slack + 1e-28 * a[0]
    assert np.isfinite(cb[0]) and abs(c[0] - want) <= cb[0] + slack
    assert np.isfinite(eb[0]) and abs(e[0] - want) <= eb[0] + slack
    assert cb[0] <= 1e4 * 256.0 * N * EPS * a[0]
    assert eb[0] <= 8 * EPS * (abs(e[0].real) + abs(e[0].imag)) + 1e-23 * a[0]


@pytest.mark.parametrize("N", [14, 16, 18])
@pytest.mark.parametrize("func", ["haf", "lhaf"])
def test_kappa_sum_matches_the_power_trace_terms(ext, oracle, func, N):
    A = rng_symmetric(3, N, 60 * N, 0.5)
    v, a = getattr(ext, f"{func}_kappa")(A)
    assert np.array_equal(v, getattr(ext, func)(A))
    assert rel_err(a, getattr(oracle, f"{func}_abs")(A)).max() < 1e-9


@pytest.mark.parametrize("N", SIDES)
def test_closed_forms(ext, N):
    """All ones (double factorial, telephone numbers), a diagonal loop hafnian
    (the product; its subset terms reach 1e11 times that at N = 24) and zero."""
    def fp64_close(func, A, want):
        v, a = getattr(ext, f"{func}_kappa")(A[None])
        assert abs(v[0] - want) <= 256.0 * N * EPS * a[0], (func, v[0], want)

    J = np.ones((N, N))
    want = math.prod(range(N - 1, 0, -2))
    fp64_close("haf", J, want)
    assert ext.haf_dd(J[None])[0] == pytest.approx(want, rel=1e-15)
    t = [1, 1]
    for k in range(2, N + 1):
        t.append(t[-1] + (k - 1) * t[-2])
    fp64_close("lhaf", J, t[N])
    assert ext.lhaf_dd(J[None])[0] == pytest.approx(t[N], rel=1e-15)
    d = np.linspace(0.5, 1.5, N)
    fp64_close("lhaf", np.diag(d), np.prod(d))
    z = np.zeros((1, N, N))
    for name in ("haf", "lhaf", "haf_dd", "lhaf_dd"):
        assert getattr(ext, name)(z)[0] == 0
    assert ext.haf_certified(z)[1][0] <= 1e-290 and ext.lhaf_dd_certified(z)[1][0] <= 1e-290


@pytest.mark.parametrize("func", ["haf", "lhaf"])
@pytest.mark.parametrize("N", [14, 18])
def test_value_independent_of_the_batch(ext, func, N):
    A = rng_symmetric(21, N, 910 + N)
    for tier in ("", "_dd"):
        full = getattr(ext, func + tier)(A)
        for idx in ([0], [20, 3], list(range(20, -1, -3))):
            assert np.array_equal(getattr(ext, func + tier)(A[idx]), full[idx])
