"""Small host calls run on pinned memory that the kernel reads and writes itself:
consecutive calls of changing sizes (across the size up to which that is done),
and calls from several threads, return what the batch engine returns."""
import sys
import threading
from pathlib import Path

import numpy as np
import pytest

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "gbskernels_amd" / "ext"))
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ext():
    import gbskernels_ext
    return gbskernels_ext


def stack(func, n, B, rng):
    A = (rng.standard_normal((B, n, n)) + 1j * rng.standard_normal((B, n, n))) / n ** 0.5
    return A if func == "perm" else (A + A.transpose(0, 2, 1)) / 2


def expect(func, tier, A):
    from gbskernels_amd.serving import Batch
    with Batch(use_graphs=False) as b:
        return b.run([(func, tier, M) for M in A])


# (n, B) below, at and above 2^20 bytes of matrices, values and auxiliaries
SIZES = [(8, 16), (1, 1), (12, 450), (12, 451), (12, 455), (16, 255), (16, 256), (2, 3), (8, 1010), (6, 1761), (10, 7)]


@pytest.mark.parametrize("func", ["perm", "haf", "lhaf"])
@pytest.mark.parametrize("tier", ["fp64", "kappa", "certified", "dd", "dd_certified"])
def test_host_calls_of_changing_sizes(ext, func, tier):
    rng = np.random.default_rng(17)
    aux = tier in ("kappa", "certified", "dd_certified")
    f = getattr(ext, func + ("" if tier == "fp64" else "_" + tier))
    for n, B in SIZES:
        n = n + n % 2 if func != "perm" else n
        B = B if n <= 8 or "dd" not in tier else min(B, 40)
        print(f"direct {func} {tier} n={n} B={B}", flush=True)
        for _ in range(2):  # the same place, other data
            A = stack(func, n, B, rng)
            v, a = expect(func, tier, A)
            r = f(A)
            assert np.array_equal(r[0] if aux else r, v)
            if aux:
                assert np.array_equal(r[1], a)


def test_host_calls_from_threads(ext):
    rng = np.random.default_rng(18)
    work = [(f, stack(f, n, B, rng)) for f in ("perm", "haf") for n, B in ((4, 5), (8, 33), (12, 64), (12, 500))]
    want = [getattr(ext, f)(A) for f, A in work]
    bad = []

    def run(k):
        for i in range(20):
            f, A = work[(i + k) % len(work)]
            if not np.array_equal(getattr(ext, f)(A), want[(i + k) % len(work)]):
                bad.append((k, i))

    ts = [threading.Thread(target=run, args=(k,)) for k in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad
