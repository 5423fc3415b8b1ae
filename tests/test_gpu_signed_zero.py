"""Signs of zero of the velocity against the oracle: walls that hold their component at -0, whose nodes
keep their velocity in the sweep across the wall, on meshes of each dual sweep's variants."""
import numpy as np
import pytest

from mahyco_amd import types as T
from tests.test_gpu_sweeps import moving_tube

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(17, 12), (65, 34), (6, 9, 35), (1, 7, 4), (66, 3, 5)], ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("sweep", ["", "tile", "flat"])
def test_velocity_keeps_the_sign_of_zero(n, sweep, monkeypatch):
    from mahyco_amd.lib import GpuCase
    from oracle.pyoracle import OracleCase
    monkeypatch.setenv("MAHYCO_SWEEP", sweep)
    c = moving_tube(n, 1)
    c.bcs = [(s, t, -0.) for s, t, _ in c.bcs]
    g, o = GpuCase(c), OracleCase(c, pow_mode=1, threads=4)
    assert g.run(7) == o.run(7)
    for d in range(c.dim):
        a, b = g.get(T.MH_N_VELOCITY, -1, d), o.get(T.MH_N_VELOCITY, -1, d)
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64)), d
    assert np.signbit(b[b == 0.]).any()
