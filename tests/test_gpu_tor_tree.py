"""Torontonians of 6 and more modes (leading modes in lane registers, middle
modes in LDS and registers): the torontonian of a direct sum is the product of
its parts', under any order of the modes, so values must agree within the
certified bounds of the three evaluations. Mode counts at the edges of the
split: no trailing mode, no leading mode, the first and the largest number of
leading modes, for the binary64 and the double-double families."""
import sys
from pathlib import Path

import numpy as np
import pytest

from physics import threshold_O

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "gbskernels_amd" / "ext"))
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ext():
    import gbskernels_ext
    return gbskernels_ext


def parts_and_sums(nm, B, rng):
    """B pairs of physical O and their direct sums in random mode orders."""
    n1 = nm // 2
    P = [np.stack([threshold_O(n, rng, eta=0.7) for _ in range(B)]).astype(np.complex128) for n in (n1, nm - n1)]
    S = np.zeros((B, 2 * nm, 2 * nm), np.complex128)
    for b in range(B):
        order = rng.permutation(nm)
        for n, at, Q in ((n1, order[:n1], P[0]), (nm - n1, order[n1:], P[1])):
            idx = np.r_[at, nm + at]
            S[b][np.ix_(idx, idx)] = (Q[b] + Q[b].T) / 2
        for k in (0, 1):
            P[k][b] = (P[k][b] + P[k][b].T) / 2
    return P[0], P[1], S


@pytest.mark.parametrize("family,nm", [("fp64", n) for n in (6, 7, 10, 11, 12, 13, 17, 20)]
                         + [("dd", n) for n in (6, 7, 8, 9, 10, 12, 14)])
def test_direct_sum_is_the_product(ext, family, nm):
    print(f"tor direct sum {family} nm={nm}", flush=True)
    cert = ext.tor_certified if family == "fp64" else ext.tor_dd_certified
    plain = ext.tor if family == "fp64" else ext.tor_dd
    A, C, S = parts_and_sums(nm, 5 if nm <= 14 else 2, np.random.default_rng(900 + nm))
    (va, ea), (vc, ec), (vs, es) = cert(A), cert(C), cert(S)
    assert np.array_equal(vs, plain(S))
    assert np.all(np.isfinite(es))
    prod = va * vc
    bound = es + abs(va) * ec + abs(vc) * ea + ea * ec + 4 * 2.0 ** -53 * abs(prod)
    assert np.all(abs(vs - prod) <= bound)


@pytest.mark.parametrize("nm,mode", [(6, 0), (6, 5), (8, 4), (12, 0), (12, 1), (12, 6), (12, 11)])
def test_off_domain_mode_is_refused(ext, nm, mode):
    """One non-positive pivot, in a leading, middle or trailing mode."""
    _, _, S = parts_and_sums(nm, 3, np.random.default_rng(950 + nm))
    good, _ = ext.tor_certified(S)
    S[1, mode, mode] = 1.5
    v, e = ext.tor_certified(S)
    assert np.isinf(e[1]) and np.all(np.isfinite(e[[0, 2]]))
    assert np.array_equal(v[[0, 2]], good[[0, 2]])
    assert np.isnan(ext.tor_dd(S)[1])
