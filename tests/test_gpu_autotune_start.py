"""The autotuner starts from the variant in place: a case that reaches its final time after the first
candidate keeps its variant (the tuner's results never replace it untimed)."""
import pytest

from mahyco_amd import types as T
from tests.test_gpu_sweeps import moving_tube

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,remap", [((13, 11, 9), False), ((14, 11, 9), True), ((29, 23), True), ((31, 23), False)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else "remap" if v else "lagrange")
def test_variant_in_place_is_the_first_candidate(n, remap):
    from mahyco_amd.lib import GpuCase
    c = moving_tube(n, 1, with_projection=remap)
    g = GpuCase(c)
    assert g.run(15) == T.MH_OK  # one candidate: 6 iterations untimed, 6 timed
    c.final_time = g.time
    g.close()
    g = GpuCase(c)
    v = g.variant
    assert g.autotune(6)[0] == v
    assert g.variant == v
    assert g.iteration <= 16
    g.close()
