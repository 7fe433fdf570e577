"""Torontonian values and bounds of 6 and more modes are the bits of the general
workgroup kernels they replaced (golden/make_tor_bits.py), and both middle walks
agree bit for bit at every mode count that has both."""
import ctypes
import importlib.util
import json
from pathlib import Path

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
GOLDEN = Path(__file__).resolve().parent / "golden"
WANT = json.loads((GOLDEN / "tor_bits.json").read_text())
spec = importlib.util.spec_from_file_location("make_tor_bits", GOLDEN / "make_tor_bits.py")
make = importlib.util.module_from_spec(spec)
spec.loader.exec_module(make)


@pytest.mark.parametrize("nm", make.MODES)
def test_batched_bits(nm):
    print(f"tor bits nm={nm}", flush=True)
    assert make.evaluate(nm) == WANT["batched"][str(nm)]


@pytest.mark.parametrize("nm", make.SINGLE)
def test_single_bits(nm):
    print(f"tor single bits nm={nm}", flush=True)
    assert make.evaluate_single(nm) == WANT["single"][str(nm)]


@pytest.mark.parametrize("nm", [1, 2, 3, 4, 5])
def test_both_walks_agree(nm):
    from gbskernels_amd import _lib
    L = _lib.lib()
    print(f"tor walks nm={nm}", flush=True)
    saved = []
    for fam in (0, 1):
        g, b = ctypes.c_int(), ctypes.c_int()
        _lib.check(L.gbs_tor_get_schedule(fam, ctypes.byref(g), ctypes.byref(b)), "get_schedule")
        saved.append((g.value, b.value))
    try:
        res = []
        for bfs in (0, 32):
            for fam in (0, 1):
                _lib.check(L.gbs_tor_set_schedule(fam, 0, bfs), "set_schedule")
            res.append(make.evaluate(nm))
        assert res[0] == res[1]
        values = np.array([int(w, 16) for w in res[0]["fp64"]], np.uint64).view(np.float64)
        assert np.all(np.isfinite(values))
    finally:
        for fam, (g, b) in enumerate(saved):
            _lib.check(L.gbs_tor_set_schedule(fam, g, b), "set_schedule")
