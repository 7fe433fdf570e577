"""Writes tor_bits.json: torontonian values, kappa sums and certified bounds, as bits, of
the general workgroup kernels (commit ab52598, before the register kernel of 6 and
more modes), run on an MI355X with GBSK_LIB naming that build's library."""
import json
import sys
from pathlib import Path

import numpy as np

HERE = Path(__file__).resolve().parent
ROOT = HERE.parent.parent
for p in (ROOT, ROOT / "tests", ROOT / "gbskernels_amd" / "ext"):
    sys.path.insert(0, str(p))

# no trailing modes (6), every trailing count, no and 1 .. 9 leading modes
MODES = [6, 7, 8, 9, 10, 11, 12, 13, 14, 16, 18, 20]
SINGLE = [12, 17, 22, 24]


def stack(nm):
    """two symmetric O with I - O positive definite; no linear algebra, so the same bits everywhere"""
    G = np.random.default_rng(40000 + nm).uniform(-1.0, 1.0, (2, 2 * nm, 2 * nm))
    return (G + G.transpose(0, 2, 1)) * (0.25 / (2 * nm) ** 0.5)


def words(x):
    """bits of the real numbers in x, the real parts of complex ones"""
    return [f"{w:016x}" for w in np.ascontiguousarray(np.real(x), np.float64).view(np.uint64).ravel()]


def evaluate(nm):
    import gbskernels_ext as ext
    O = stack(nm).astype(np.complex128)
    res = {"fp64": (ext.tor(O),), "kappa": ext.tor_kappa(O), "certified": ext.tor_certified(O), "dd": (ext.tor_dd(O),),
           "dd_certified": ext.tor_dd_certified(O)}
    return {k: [w for x in v for w in words(x)] for k, v in res.items()}


def evaluate_single(nm):
    import gbskernels_ext as ext
    O = stack(nm)[0]
    res = {"single_ddcertified": ext.tor_single_ddcertified(O, 4), "single": (ext.tor_single(O, 4),), "single_certified": ext.tor_single_certified(O, 4)}
    return {k: [w for x in v for w in words(np.atleast_1d(x))] for k, v in res.items()}


if __name__ == "__main__":
    out = {"batched": {str(n): evaluate(n) for n in MODES}, "single": {str(n): evaluate_single(n) for n in SINGLE}}
    Path(sys.argv[1]).write_text(json.dumps(out, indent=0) + "\n")
