"""Members of an ensemble on both sides of the lines at which their cell sweeps change, bit for bit against
the oracle: the segments of the marching sweeps on small meshes, the presence bytes of 3D members."""
import pytest

from tests.helpers import bitwise_equal, fields
from tests.test_gpu_sweeps import moving_tube

pytestmark = pytest.mark.gpu


class Member:
    def __init__(self, e, slot):
        self.e, self.slot = e, slot

    def get(self, field, env=-1, comp=0):
        return self.e.get(self.slot, field, env, comp)


def one_environment(c):
    from mahyco_amd import types as T
    c.envs, c.cas_model, c.cas_test = c.envs[:1], T.MH_CASE_SOD, 3
    return c


@pytest.mark.parametrize("m", [1, 2])
@pytest.mark.parametrize("dim", [2, 3])
def test_small_members(dim, m):
    sizes = {2: [(2, 2), (5, 7), (12, 13), (3, 331), (333, 3), (25, 40), (63, 65), (64, 64), (65, 64)],
             3: [(2, 2, 2), (3, 5, 7), (8, 9, 10), (15, 16, 17), (16, 16, 16), (2, 33, 17), (17, 16, 16)]}[dim]
    cases = [moving_tube(n, 1) for n in sizes]
    check([one_environment(c) for c in cases] if m == 1 else cases, m, dim)


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_presence_bytes(seed):
    check([moving_tube(n, seed) for n in ((15, 16, 17), (16, 15, 17), (2, 40, 40), (40, 40, 2), (99, 100, 101),
                                          (100, 100, 100))], 2, 3)


def check(cases, m, dim):
    from mahyco_amd.lib import Ensemble
    from oracle.pyoracle import OracleCase
    e = Ensemble(len(cases), 8 << 30)
    slots = [e.add(c) for c in cases]
    e.step(7)
    e.synchronize()
    bad = []
    for c, s in zip(cases, slots):
        o = OracleCase(c, pow_mode=1, threads=4)
        o.run(7)
        a, b = fields(Member(e, s), m, dim), fields(o, m, dim)
        bad += [(c.n, k) for k in a if not bitwise_equal(a[k], b[k])]
        o.close()
    e.close()
    assert not bad, bad
