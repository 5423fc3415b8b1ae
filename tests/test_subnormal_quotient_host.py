"""Subnormal quotients of the shared-denominator division on the host, bit for bit against plain
division: exact ties between two subnormals, their neighbours, quotients that underflow to zero, and
ordinary operands with quotients on both sides of the smallest normal number."""
import numpy as np

from tests.test_signed_zero_host import _run, checker  # noqa: F401


def test_subnormal_quotients(checker):  # noqa: F811
    rng = np.random.default_rng(20261206)
    n = 40000
    # a = b (k + 1/2) 2^-1074 with short significands: exact, the quotient a tie
    k = rng.integers(0, 1 << 20, n).astype(float)
    b = (rng.integers(0, 1 << 20, n) | 1).astype(float)
    s = rng.integers(53, 400, n)
    sign = rng.choice([-1., 1.], n)
    ties = np.stack([sign * np.ldexp(b * (2 * k + 1), s - 1075), np.ldexp(b, s)], 1)
    near = ties.copy()
    near[:, 0] = np.nextafter(near[:, 0], rng.choice([-np.inf, np.inf], n))
    m = rng.choice([-1., 1.], n) * rng.uniform(1., 2., n)
    wide = np.stack([np.ldexp(m, rng.integers(-960, -300, n)), np.ldexp(rng.uniform(1., 2., n), rng.integers(60, 1000, n))], 1)
    edge = np.stack([np.ldexp(m, rng.integers(-900, -800, n)), np.ldexp(rng.uniform(1., 2., n), rng.integers(120, 180, n))], 1)
    assert _run(checker, np.concatenate([ties, near, wide, edge]))[0] == 0
