"""Zeros in the shared-denominator quotients and the one-division limited gradients of the sweeps, on
the host as the kernels are built (g++, -ffp-contract=off): the bits of plain division, the sign of a
zero included, and the values of the two-sided limiter formula (UtilesRemap.cc:325-357)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("zero") / "signed_zero_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", os.path.join(HERE, "host", "signed_zero_check.cpp"),
                    "-o", exe], check=True)
    return exe


def _run(checker, p):
    p = np.ascontiguousarray(p)
    text = "\n".join("%x %x" % (a, b) for a, b in p.view(np.uint64))
    r = subprocess.run([checker], input=text, capture_output=True, text=True, check=True)
    out = tuple(map(int, r.stdout.split()))
    assert out[0] == len(p)
    return out[1:]


def test_signed_zeros(checker):
    """Every pair of zeros, ordinary numbers, subnormals, the ends of the range, infinities and NaN,
    and zeros against random numbers."""
    rng = np.random.default_rng(20261205)
    special = np.array([0., 1., 2., 3., .5, 5e-324, 1e-310, 2.2e-308, 1e-300, 1e-160, 1e160, 1.7e308, np.inf, np.nan])
    special = np.concatenate([special, -special])
    gx, gy = np.meshgrid(special, special)
    r = rng.choice([-1., 1.], 20000) * np.ldexp(rng.uniform(1., 2., 20000), rng.integers(-60, 60, 20000))
    z = rng.choice([0., -0.], 20000)
    assert _run(checker, np.concatenate([np.stack([gx.ravel(), gy.ravel()], 1), np.stack([z, r], 1),
                                         np.stack([r, z], 1)])) == (0, 0)
