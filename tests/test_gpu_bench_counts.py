"""bench.py's executed work: with the kernels' counted FP64 instructions no cell runs
above the FP64 peak or the issue rate (counts of other kernels did)."""
import json
import subprocess
import sys
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu
ROOT = Path(__file__).resolve().parent.parent
CELLS = ["haf_fp64_n16", "haf_fp64_n24", "lhaf_fp64_n16", "lhaf_fp64_n24", "tor_fp64_nm8", "tor_fp64_nm12",
         "tor_fp64_nm16"]


def test_executed_rates_are_possible():
    print("bench cells", flush=True)
    r = subprocess.run([sys.executable, str(ROOT / "bench.py"), "--cells", ",".join(CELLS), "--reps", "3"],
                       capture_output=True, text=True, timeout=100, check=True)
    cells = json.loads(r.stdout.strip().splitlines()[-1])["cells"]
    for name in CELLS:
        c = cells[name]
        assert 0.05 < c["fp64_issue_frac"] < 0.8, (name, c)
        assert 0.0 < c["tflops_executed"] < 0.8 * 78.6, (name, c)
