"""Fields read back through the pinned slots, against the oracle: one slot (up to 256 KB), a ring of
four with one thread and with several, more chunks than slots, and several cases read at once."""
import threading

import pytest

from tests.helpers import bitwise_equal, fields
from tests.test_gpu_sweeps import moving_tube

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(7, 5), (181, 181), (182, 181), (513, 512), (1100, 700), (1450, 1500), (2, 3, 4)],
                         ids=lambda n: "x".join(map(str, n)))
def test_fields_of_every_size(n):
    from mahyco_amd.lib import GpuCase
    from oracle.pyoracle import OracleCase
    c = moving_tube(n, 1)
    g, o = GpuCase(c), OracleCase(c, pow_mode=1, threads=4)
    assert g.run(3) == o.run(3)
    a, b = fields(g, 2, c.dim), fields(o, 2, c.dim)
    assert not [k for k in a if not bitwise_equal(a[k], b[k])]


def test_cases_read_by_several_threads():
    from mahyco_amd.lib import GpuCase
    sizes = [(60, 40), (700, 500), (1200, 900), (181, 182)]
    gs = [GpuCase(moving_tube(n, 1)) for n in sizes]
    for g in gs:
        g.run(3)
    alone = [fields(g, 2, 2) for g in gs]
    got = [None] * len(gs)

    def read(i):
        for _ in range(3):
            got[i] = fields(gs[i], 2, 2)
    ts = [threading.Thread(target=read, args=(i,)) for i in range(len(gs))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for a, b in zip(alone, got):
        assert not [k for k in a if not bitwise_equal(a[k], b[k])]
