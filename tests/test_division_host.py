"""The shared-denominator division and the one-division limiters of the sweeps on the host (g++,
-ffp-contract=off as the kernels are built), bit for bit against plain division and the two-sided
limiter formula (UtilesRemap.cc:108-120, 325-357).  Operands: random significands over wide and
narrow exponent ranges, quotients next to rounding midpoints and to the limiters' thresholds,
small integers, equal and opposite pairs, and every pair of zeros, infinities, NaN, subnormals
and the ends of the range."""
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def _pairs(rng):
    def rnd(n, lo, hi):
        return rng.choice([-1., 1.], n) * np.ldexp(rng.uniform(1., 2., n), rng.integers(lo, hi + 1, n))
    out = [np.stack([rnd(200000, -2, 2), rnd(200000, -2, 2)], 1), np.stack([rnd(100000, -300, 300), rnd(100000, -300, 300)], 1),
           np.stack([rnd(20000, -1074, 1000), rnd(20000, -1074, 1000)], 1),
           # small numerators, whose remainders underflow
           np.stack([rnd(300000, -1074, -900), rnd(300000, -60, 10)], 1)]
    # x = RN(b (k + 1/2 ulp)): quotients next to midpoints
    b, k = rnd(100000, -1, 1), rnd(100000, -1, 1)
    for m in (k + np.spacing(k) / 2, k):
        x = b * m
        for d in (-1, 0, 1):
            out.append(np.stack([x + d * np.spacing(x), b], 1))
    # ratios at and next to 1/2, 1 and 2
    y = rnd(30000, -3, 3)
    for f in (.5, 1., 2., -1., -2.):
        for d in (-2, -1, 0, 1, 2):
            x = f * y
            out.append(np.stack([x + d * np.spacing(x), y], 1))
    i = rng.integers(-9, 10, (50000, 2)).astype(float)
    out.append(i)
    one_ulp = 1. + np.arange(-40, 41) * 2. ** -53
    gx, gy = np.meshgrid(one_ulp, one_ulp)
    out.append(np.stack([gx.ravel(), gy.ravel()], 1))
    special = np.array([0., -0., np.inf, -np.inf, np.nan, 5e-324, -5e-324, 2.2e-308, 1e-300, -1e-300, 1.7e308, -1.7e308,
                        1e-160, 1e160, 1., -1., 2., .5, 3.])
    gx, gy = np.meshgrid(special, special)
    out.append(np.stack([gx.ravel(), gy.ravel()], 1))
    return np.concatenate(out)


def test_shared_division_and_limiters_bitwise(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "division_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", os.path.join(HERE, "host", "division_check.cpp"),
                    "-o", exe], check=True)
    p = np.ascontiguousarray(_pairs(np.random.default_rng(20261205)))
    text = "\n".join("%x %x" % (a, b) for a, b in p.view(np.uint64))
    r = subprocess.run([exe], input=text, capture_output=True, text=True, check=True)
    pairs, div, lim = map(int, r.stdout.split())
    assert pairs == len(p)
    assert div == 0
    assert lim == 0
