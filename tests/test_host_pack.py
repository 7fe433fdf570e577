"""pack() works column by column; it must give what the loop over items gives,
and refuse with the same error, whatever the items hold."""
import numpy as np
import pytest

from gbskernels_amd import serving

rng = np.random.default_rng(0)


def M(n, m=None):
    return rng.standard_normal((n, m or n)) + 1j * rng.standard_normal((n, m or n))


CASES = [
    [], (("perm", "fp64", M(3)),), [("perm", "fp64", M(0)), ("perm", "dd", M(2))],
    [("perm", "fp64", M(3)), ("lhaf", "dd", M(5)), ("haf", "kappa", M(4).real), ("tor", "auto", M(4))],
    [("perm", "fp64", M(4).T), ("haf", "fp64", [[0, 1], [1, 0]]), ("lhaf", "fp64", M(6)[::2, ::2])],
    [("haf", "fp64", M(3)), ("lhaf", "fp64", M(1)), ("perm", "fp64", M(2).astype(np.complex64))],
    [("perm", "fp64", M(3)), ("tor", "fp64", M(5)), ("x", "fp64", M(2))],
    [("perm", "fp64", M(3, 2)), ("x", "fp64", 1)], [("x", "fp64", 1), ("perm", "fp64", M(3, 2))],
    [("perm", "zz", M(1))], [("perm", "fp64", 3.0)], [("perm", "fp64")], [("perm", "fp64", "abc")],
    [("perm", "fp64", M(2), 1)], [(["perm"], "fp64", M(2))],
]


@pytest.mark.parametrize("k", range(len(CASES)))
def test_pack_equals_the_loop_over_items(k):
    res = []
    for f in (serving.pack, serving._pack_items):
        try:
            res.append(f(CASES[k]))
        except Exception as e:
            res.append((type(e), str(e)))
    a, b = res
    if isinstance(b[0], type):
        assert a == b
        return
    for x, y in zip(a, b):
        assert x.dtype == y.dtype and x.shape == y.shape and x.flags.c_contiguous and np.array_equal(x, y)
