"""Several host threads read fields of one case, and of the members of one ensemble: each read gives
what a read alone gives.  A process's first reads give what its later ones do."""
import os
import subprocess
import sys
import threading

import pytest

from mahyco_amd import types as T
from tests.helpers import bitwise_equal
from tests.test_gpu_sweeps import moving_tube

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


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


# A process's first reads take the plain route (copies and a loop over the cells), later ones of values
# formed per cell the pinned one: in a process of its own, both against the oracle and each other.
FIRST_READS = """
from mahyco_amd import cases, types as T
from mahyco_amd.lib import GpuCase
from oracle.pyoracle import OracleCase
from tests.helpers import bitwise_equal, fields
from tests.test_gpu_sweeps import moving_tube

def more(g, m):
    out = {("materiau",): g.get(T.MH_F_MATERIAU), ("mass fraction",): g.get(T.MH_F_MASS_FRACTION)}
    for f in (T.MH_F_CELL_VOLUME, T.MH_F_SOUND_SPEED, T.MH_F_PSEUDO_VISCOSITY):
        for k in range(-1, m):
            out[f, k] = g.get(f, k)
    return out

triple = cases.bitriplepoint()
for c in (moving_tube((7, 5), 1), moving_tube((2, 3, 4), 1), triple, moving_tube((181, 90), 1)):
    m = len(c.envs)
    g, o = GpuCase(c), OracleCase(c, pow_mode=1, threads=4)
    assert g.run(5) == o.run(5)
    first = {**fields(g, m, c.dim), **more(g, m)}
    for _ in range(30):
        g.get(T.MH_F_DENSITY, 0)
    later = {**fields(g, m, c.dim), **more(g, m)}
    ref = fields(o, m, c.dim)
    bad = [k for k in first if not bitwise_equal(first[k], later[k])] + \\
          [k for k in ref if not bitwise_equal(first[k], ref[k])]
    assert not bad, (c.name, bad)
    g.close()
print("first reads ok")
"""


def test_first_reads_of_a_process():
    r = subprocess.run([sys.executable, "-c", FIRST_READS], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "first reads ok" in r.stdout, r.stderr[-2000:]
