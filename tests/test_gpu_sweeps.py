"""The remap sweeps at the edges of their launch shapes, bit for bit against the oracle.

Meshes of one to a few cells per direction, one more or less than a row segment (60 lanes), a
tile (64 x 16) or a marching segment, and directions one cell wide, which are not swept: every
number of sweeps per remap (one, two, three) and every rotation of their order.  A moving tube
with walls sends material through every face; the interface lies inside a cell, so pure and
mixed cells meet."""
import numpy as np
import pytest

from mahyco_amd import cases
from mahyco_amd import types as T
from tests.helpers import bitwise_equal, fields

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (3, 17, 4), (61, 5, 3), (122, 3, 2), (5, 1, 6), (1, 7, 4), (4, 3, 1), (1, 1, 5), (7, 33, 2),
          (64, 4, 18), (65, 2, 17), (6, 9, 35)]
FLAT = [(2, 2), (3, 17), (61, 18), (122, 5), (1, 9), (8, 1), (65, 34)]


def moving_tube(n, seed, **kw):
    rng = np.random.default_rng(seed)
    c = cases.riemann2d(n[0], n[1], rng, stiffened=bool(seed % 2), name="moving_%s_%d" % ("x".join(map(str, n)), seed))
    if len(n) == 3:
        c.dim, c.n, c.length, c.bcs = 3, n, (1., 1., 1.), list(cases.WALLS_3D)
    c.interface_axis = seed % len(n)
    c.limiter = (T.MH_MINMOD, T.MH_SUPERBEE, T.MH_VANLEER)[seed % 3]
    for e in c.envs:
        e.vitesse_initiale = (.4, -.3, .2)
    for k, v in kw.items():
        setattr(c, k, v)
    return c


def check(c, iterations=13):
    from mahyco_amd.lib import GpuCase
    from oracle.pyoracle import OracleCase
    g, o = GpuCase(c), OracleCase(c, pow_mode=1, threads=4)
    st = g.run(iterations)
    assert st == o.run(iterations) and g.iteration == o.iteration
    assert (g.time, g.deltat) == (o.time, o.deltat)
    a, b = fields(g, len(c.envs), c.dim), fields(o, len(c.envs), c.dim)
    bad = [k for k in a if not bitwise_equal(a[k], b[k])]
    g.close()
    o.close()
    assert not bad, bad


# the variants a mesh takes by its size, and at every size those of the large meshes (tiles,
# marching segments) and one thread per item
@pytest.mark.parametrize("sweep,node", [("", ""), ("tile", "tiled"), ("flat", "flat")])
@pytest.mark.parametrize("seed", [0, 1, 2])
@pytest.mark.parametrize("n", SHAPES + FLAT, ids=lambda n: "x".join(map(str, n)))
def test_sweeps_at_launch_shape_edges(n, seed, sweep, node, monkeypatch):
    monkeypatch.setenv("MAHYCO_SWEEP", sweep)
    monkeypatch.setenv("MAHYCO_NODE_KERNEL", node)
    check(moving_tube(n, seed))


@pytest.mark.parametrize("n", [(181, 20), (300, 100), (31, 30, 29), (62, 40, 20)], ids=lambda n: "x".join(map(str, n)))
def test_slots_shared_out(n):
    """Meshes around the lines between one, two, four and all slots per thread."""
    check(moving_tube(n, 2), iterations=5)


@pytest.mark.parametrize("n", [(3, 17, 4), (5, 1, 6), (1, 1, 5), (61, 18)], ids=lambda n: "x".join(map(str, n)))
def test_total_energy_reads_the_last_sweeps_mass(n):
    check(moving_tube(n, 1, conservation_energie_totale=True))


@pytest.mark.parametrize("seed", [0, 1])
@pytest.mark.parametrize("n", SHAPES + FLAT, ids=lambda n: "x".join(map(str, n)))
def test_order3_segments(n, seed):
    """The order-3 sweep at odd and even line lengths, lines shorter than its stencil included."""
    check(moving_tube(n, seed, ordre_projection=3))


def test_order3_three_materials():
    check(moving_tube((61, 18), 2, ordre_projection=3, envs=[cases.Env(d, p, 1.4, vitesse_initiale=(.4, -.3, 0.))
                                                             for d, p in ((1., 1.), (.5, .3), (.2, .1))]))


@pytest.mark.parametrize("debar", [0, 1, 2])
@pytest.mark.parametrize("n", [(3, 17, 4), (1, 7, 4), (61, 18), (2, 2)], ids=lambda n: "x".join(map(str, n)))
def test_pente_borne_groups(n, debar):
    """Pente-borne fluxes with each debar fix: every group of environments on its own."""
    check(moving_tube(n, debar, pente_borne=True, debar_fix=debar, pente_borne_mixte=debar != 2,
                      limiter=T.MH_SUPERBEE_G if debar else T.MH_MINMOD, simple_pente=debar == 1,
                      limiter_pure=T.MH_VANLEER_G))


@pytest.mark.parametrize("limiter", [T.MH_MINMOD_G, T.MH_VANLEER_G, T.MH_ARITHMETIC_G, T.MH_ULTRABEE_G])
def test_generalised_limiters(limiter):
    check(moving_tube((9, 5, 4), 1, limiter=limiter))


@pytest.mark.parametrize("name", ["served114", "served162"])
def test_emptying_cells_with_presence_bytes(name, monkeypatch):
    """Runs whose cells empty out (phi of an empty cell, zero denominators), with the sweeps that
    skip the slots of environments a stencil does not hold."""
    from tests.test_gpu_paths import test_full_size_bitwise_vs_oracle
    monkeypatch.setenv("MAHYCO_SWEEP", "tile")
    test_full_size_bitwise_vs_oracle(name)


@pytest.mark.parametrize("sweep", ["tile", "flat"])
def test_presence_bytes_three_materials(sweep, monkeypatch):
    monkeypatch.setenv("MAHYCO_SWEEP", sweep)
    c = cases.bitriplepoint()
    c.n = (130, 67, 1)
    check(c, iterations=60)


def test_presence_bytes_over_variants_and_checkpoint(tmp_path, monkeypatch):
    """Sweep variants that keep the presence bytes and variants that do not, in turn on one case, and
    a restart in between."""
    from mahyco_amd.lib import GpuCase
    from oracle.pyoracle import OracleCase
    monkeypatch.setenv("MAHYCO_SWEEP", "tile")
    c = moving_tube((70, 33), 1)
    g, o = GpuCase(c), OracleCase(c, pow_mode=1, threads=4)
    v = g.variant
    for k, code in enumerate((v, v | 16, v)):
        g.set_variant(code)
        g.run(7)
        o.run(7)
        if k == 1:
            g.checkpoint_write(tmp_path / "dump")
            g.run(3)
            g.checkpoint_read(tmp_path / "dump")
    a, b = fields(g, 2, 2), fields(o, 2, 2)
    assert not [k for k in a if not bitwise_equal(a[k], b[k])]


# node kernels: blocks of 64 nodes (64, 65 and 128 of them), tiles of 31 x 7 columns and one more,
# depths that end on, before and after the last node plane; then the remap's other Lagrange steps
@pytest.mark.parametrize("variant", [0, 1, 2, 3])
@pytest.mark.parametrize("kw", [{}, dict(with_projection=False)], ids=["remap", "lagrange"])
@pytest.mark.parametrize("n", [(3, 3, 3), (4, 12, 1), (7, 7, 1), (30, 6, 11), (31, 7, 12), (32, 8, 15), (5, 3, 16)],
                         ids=lambda n: "x".join(map(str, n)))
def test_node_kernels_at_block_edges(n, kw, variant):
    from mahyco_amd.lib import GpuCase
    from oracle.pyoracle import OracleCase
    c = moving_tube(n, variant, **kw)
    g, o = GpuCase(c), OracleCase(c, pow_mode=1, threads=4)
    g.set_variant(variant)
    assert g.run(7) == o.run(7)
    a, b = fields(g, 2, 3), fields(o, 2, 3)
    assert not [k for k in a if not bitwise_equal(a[k], b[k])]


# the marching cell sweeps: lines shorter than a segment, segments of unequal length, wavefronts
# that span lines, one environment (2D, 3D) and two (2D, above with MAHYCO_SWEEP=tile)
@pytest.mark.parametrize("sweep", ["tile", "flat"])
@pytest.mark.parametrize("n", [(2, 2, 2), (5, 17, 33), (61, 16, 15), (3, 47, 1), (70, 34, 5), (2, 2), (65, 9), (7, 41)],
                         ids=lambda n: "x".join(map(str, n)))
def test_one_environment_marching_sweeps(n, sweep, monkeypatch):
    monkeypatch.setenv("MAHYCO_SWEEP", sweep)
    c = moving_tube(n, n[0] % 3)
    # a single-material tube along one of the axes
    c.envs, c.cas_model, c.cas_test = c.envs[:1], T.MH_CASE_SOD, 3 + (n[0] + n[1]) % len(n)
    check(c)


@pytest.mark.parametrize("envs", [1, 2])
@pytest.mark.parametrize("n", [(7, 41), (5, 17, 33)], ids=lambda n: "x".join(map(str, n)))
def test_csts_velocities_in_the_large_mesh_sweeps(n, envs, monkeypatch):
    monkeypatch.setenv("MAHYCO_SWEEP", "tile")
    c = moving_tube(n, 0, schema_csts=True)
    if envs == 1:
        c.envs, c.cas_model, c.cas_test = c.envs[:1], T.MH_CASE_SOD, 4
    check(c)
