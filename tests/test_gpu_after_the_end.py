"""Iterations queued beyond a run's end are no-ops and cost next to nothing beside running ones: the
blocks of a launch leave at the stop flag before they read what they would work on.  (Shares of a running
iteration, 128^3 cells alone and 8 meshes of 48^3 at once: 0.04 and 0.08; 0.23 and 0.26 where every
block reads its cells first.)"""
import time

import pytest

from tests.test_gpu_sweeps import moving_tube

pytestmark = pytest.mark.gpu


def _best(f, repeats=5):
    out = []
    for _ in range(repeats):
        t = time.perf_counter()
        f()
        out.append(time.perf_counter() - t)
    return min(out)


def test_single_mesh():
    from mahyco_amd.lib import GpuCase
    c = moving_tube((128, 128, 128), 1, final_time=1e30)
    times = []
    for end in (1e30, 1e-12):
        c.final_time = end
        g = GpuCase(c)
        g.run(6, graph=6)
        times.append(_best(lambda: g.run(24, graph=6)))
        it = g.iteration
        g.run(6, graph=6)
        assert (g.iteration == it) == (end < 1.)
        g.close()
    assert times[1] < 0.12 * times[0], times


def test_ensemble():
    from mahyco_amd.lib import Ensemble
    times = []
    for end in (1e30, 1e-12):
        e = Ensemble(8, 16 << 30)
        for i in range(8):
            assert e.add(moving_tube((48 + i, 48, 48), 1, final_time=end)) is not None
        e.step(6)

        def steps():
            e.step(24)
            e.synchronize()
        steps()
        times.append(_best(steps))
        e.close()
    assert times[1] < 0.16 * times[0], times
