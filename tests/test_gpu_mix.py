"""Multi-size launches of a mixed batch: every size a launch can carry, with
counts at the edges of a workgroup, equals the uniform call bit for bit (values
and kappa sums), eager and from a captured graph replayed with other inputs."""
import sys
from pathlib import Path

import numpy as np
import pytest

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "gbskernels_amd" / "ext"))
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ext():
    import gbskernels_ext
    return gbskernels_ext


def items_of(func, tier, counts, rng):
    out = []
    for n, c in counts.items():
        for _ in range(c):
            A = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) / max(n, 1) ** 0.5
            out.append((func, tier, A if func == "perm" else (A + A.T) / 2))
    return [out[i] for i in rng.permutation(len(out))]


def check(ext, batch, items):
    values, aux = batch.run(items)
    groups = {}
    for i, (f, t, A) in enumerate(items):
        groups.setdefault((f, t, A.shape[0]), []).append(i)
    for (f, t, n), at in groups.items():
        stack = np.stack([items[i][2] for i in at])
        if t == "kappa":
            v, a = getattr(ext, f + "_kappa")(stack)
            assert np.array_equal(aux[at], a), (f, n)
        else:
            v = getattr(ext, f)(stack)
        assert np.array_equal(values[at], v), (f, t, n)


PERM = [{0: 2, 1: 65, 2: 1, 3: 64, 4: 63, 5: 65, 6: 33, 7: 17, 8: 9, 9: 5, 10: 3, 11: 1},
        {n: 1 + n % 3 for n in range(11, 26)},
        {5: 3, 16: 9, 17: 65, 18: 8, 26: 1, 27: 1, 28: 1}]


@pytest.mark.parametrize("tier", ["fp64", "kappa"])
@pytest.mark.parametrize("graphs", [False, True])
@pytest.mark.parametrize("k", range(len(PERM)))
def test_perm_sizes_in_one_launch(ext, k, graphs, tier):
    from gbskernels_amd.serving import Batch
    print(f"perm mix {k} {tier} graphs={graphs}", flush=True)
    with Batch(use_graphs=graphs) as b:
        for seed in range(3 if graphs else 1):
            check(ext, b, items_of("perm", tier, PERM[k], np.random.default_rng(70 + 10 * k + seed)))


def test_both_tiers_and_functions_together(ext):
    from gbskernels_amd.serving import Batch
    rng = np.random.default_rng(99)
    items = []
    for tier in ("fp64", "kappa"):
        items += items_of("perm", tier, {n: 2 for n in range(1, 21)}, rng)
        items += items_of("haf", tier, {n: 3 for n in range(2, 25, 2)}, rng)
        items += items_of("lhaf", tier, {n: 3 for n in range(2, 25, 2)}, rng)
    with Batch(use_graphs=False) as b:
        check(ext, b, [items[i] for i in rng.permutation(len(items))])
