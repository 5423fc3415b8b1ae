"""The pente-borne and generalised-limiter sweeps on meshes narrower than their tiles and at the edges
of these, bit for bit against the oracle."""
import pytest

from mahyco_amd import types as T
from tests.test_gpu_sweeps import check, moving_tube

pytestmark = pytest.mark.gpu

SHAPES = [(1, 300), (2, 129), (3, 64), (5, 51), (15, 17), (31, 9), (32, 8), (33, 15), (1, 9, 40), (2, 17, 9), (3, 3, 70),
          (7, 5, 16), (31, 2, 8), (5, 40, 3)]


@pytest.mark.parametrize("n", SHAPES, ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("opt", [dict(limiter=T.MH_SUPERBEE_G), dict(limiter=T.MH_MINMOD_G, pente_borne=True, debar_fix=1)],
                         ids=["superbeeG", "pente-borne"])
def test_narrow_meshes(n, opt):
    c = moving_tube(n, 1, **opt)
    check(c, iterations=7)
