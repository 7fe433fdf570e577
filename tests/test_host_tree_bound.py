"""The certified bound of the series tree's products (tree_product, fp64), run on the
CPU and compared with exact rational arithmetic: operands that cancel in the sum,
and operands whose own bounds are as large as they are. A rule that leaves out the
product of the bounds must fail here.

The bound's own arithmetic is in round to nearest; cert_finish inflates the end
result by 1 + 2 D u for its rounding depth D, here below 64 (7 steps of 5 and the end)."""
import math
import shutil
import subprocess
from fractions import Fraction
from pathlib import Path

import pytest

from gbskernels_amd import _lib

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
CSRC = Path(_lib.__file__).parent / "csrc"
H = 7
U = Fraction(1, 2 ** 53)
SOURCE = r"""
#include <cstdio>
#include <random>
#include "haf_tree.hpp"
using namespace gbsk;
constexpr int H = 7;
int main() {
  std::mt19937_64 g(11);
  std::normal_distribution<double> n;
  for (int t = 0; t < 400; ++t) {
    // kinds: 0 plain, 1 the last products cancel the first, 2 bounds as large as the values
    const int kind = t % 3;
    cplx x[H], y[H], acc[H];
    double ex[H], ey[H], ea[H];
    for (int i = 0; i < H; ++i) {
      x[i] = cplx{n(g), n(g)};
      y[i] = cplx{n(g), n(g)};
      ex[i] = kind == 2 ? fabs(n(g)) : 0.0;
      ey[i] = kind == 2 ? fabs(n(g)) : 0.0;
    }
    if (kind == 1) {  // x_0 y_1 + x_1 y_0: equal products, opposite signs; real parts by Im x Im y
      x[0] = cplx{n(g), 1e3 * n(g)};
      y[0] = cplx{n(g), 1e3 * n(g)};
      x[1] = cplx{-x[0].re, -x[0].im};
      y[1] = y[0];
    }
    tree_product<true, H>([&](int i, cplx& a, double& e) { a = x[i]; e = ex[i]; }, y, ey, acc, ea);
    std::printf("%d", kind);
    for (int i = 0; i < H; ++i)
      std::printf(" %a %a %a %a %a %a %a %a %a", x[i].re, x[i].im, ex[i], y[i].re, y[i].im, ey[i], acc[i].re, acc[i].im, ea[i]);
    std::printf("\n");
  }
}
"""


def mul(a, b):
    return a[0] * b[0] - a[1] * b[1], a[0] * b[1] + a[1] * b[0]


def add(a, b):
    return a[0] + b[0], a[1] + b[1]


def square(a):
    return a[0] * a[0] + a[1] * a[1]


def norm(a):  # |a| from above
    return Fraction(math.sqrt(square(a))) * (1 + 4 * U)


@pytest.fixture(scope="module")
def rows(tmp_path_factory):
    d = tmp_path_factory.mktemp("bound")
    (d / "b.hip").write_text(SOURCE)
    subprocess.run([HIPCC, "--cuda-host-only", "-std=c++17", "-O1", "-ffp-contract=off", f"-I{CSRC}", "-c",
                    str(d / "b.hip"), "-o", str(d / "b.o")], check=True)
    subprocess.run([HIPCC, str(d / "b.o"), "-o", str(d / "b")], check=True)
    out = subprocess.run([str(d / "b")], check=True, capture_output=True, text=True).stdout
    res = []
    for line in out.splitlines():
        kind, *v = line.split()
        v = [Fraction(float.fromhex(q)) for q in v]
        res.append((int(kind), [v[9 * i:9 * i + 9] for i in range(H)]))
    return res


def worst_error(c, d):
    """Square of the largest |acc_d - exact| over operands moved by their bounds along one direction
    each (real or imaginary, either sign)."""
    best = Fraction(0)
    for sx in ((1, 0), (-1, 0), (0, 1), (0, -1)):
        for sy in ((1, 0), (-1, 0), (0, 1), (0, -1)):
            s = (Fraction(0), Fraction(0))
            for i in range(d + 1):
                a, b = c[i], c[d - i]
                s = add(s, mul((a[0] + sx[0] * a[2], a[1] + sx[1] * a[2]), (b[3] + sy[0] * b[5], b[4] + sy[1] * b[5])))
            best = max(best, square((s[0] - c[d][6], s[1] - c[d][7])))
    return best


def test_products_are_enclosed(rows):
    for kind, c in rows:
        for d in range(H):
            assert worst_error(c, d) <= (c[d][8] * (1 + 2 * 64 * U)) ** 2, (kind, d)


def test_a_rule_without_the_product_of_bounds_does_not_enclose(rows):
    """2u |acc_after| + |x| ey + ex |y| a step: what the products of the last level charged."""
    failed = set()
    for kind, c in rows:
        for d in range(H):
            e, acc = Fraction(0), (Fraction(0), Fraction(0))
            for i in range(d + 1):
                a, b = c[i], c[d - i]
                acc = add(acc, mul(a[:2], b[3:5]))
                e += 2 * U * norm(acc) + norm(a[:2]) * b[5] + a[2] * norm(b[3:5])
            if worst_error(c, d) > (e * (1 + 2 * 64 * U)) ** 2:
                failed.add(kind)
    assert 2 in failed
