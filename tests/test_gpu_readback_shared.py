"""Several host threads read fields of one case, and of the members of one ensemble: each read gives
what a read alone gives."""
import threading

import pytest

from mahyco_amd import types as T
from tests.helpers import bitwise_equal
from tests.test_gpu_sweeps import moving_tube

pytestmark = pytest.mark.gpu


def _together(reads, rounds=6):
    """Runs each of `reads` (functions returning an array) in its own thread, `rounds` times over,
    and returns the reads that differed from the same read alone."""
    alone = [r() for r in reads]
    wrong = []

    def work(i):
        for _ in range(rounds):
            if not bitwise_equal(reads[i](), alone[i]):
                wrong.append(i)
    ts = [threading.Thread(target=work, args=(i,)) for i in range(len(reads))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    return wrong


def test_threads_read_one_case():
    from mahyco_amd.lib import GpuCase
    g = GpuCase(moving_tube((1100, 700), 1))
    g.run(3)
    assert not _together([lambda: g.get(T.MH_F_DENSITY), lambda: g.get(T.MH_F_FRACVOL, 1),
                          lambda: g.get(T.MH_N_VELOCITY, -1, 0), lambda: g.get(T.MH_F_MATERIAU)])


def test_threads_read_one_ensemble():
    from mahyco_amd.lib import Ensemble
    e = Ensemble(3, 8 << 30)
    slots = [e.add(moving_tube(n, 1)) for n in ((60, 40), (700, 500), (1200, 900))]
    e.step(3)
    e.synchronize()
    reads = [lambda s=s, f=f, k=k: e.get(s, f, k) for s in slots for f, k in ((T.MH_F_PRESSURE, -1), (T.MH_F_DENSITY, 0))]
    assert not _together(reads)
    e.close()
