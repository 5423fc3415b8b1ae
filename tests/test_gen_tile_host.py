"""The tiles of the pente-borne / generalised-limiter sweeps (GenTile, mahyco_amd/csrc/mh_geom.h) on the
host: every cell is updated by one thread, the face ahead of it is the next row's in its block, and
narrow meshes do not launch many more threads than they have cells."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_tiles_cover_the_mesh(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "gen_tile_check")
    subprocess.run(["g++", "-O2", "-std=c++17", os.path.join(HERE, "host", "gen_tile_check.cpp"), "-o", exe], check=True)
    shapes = [(nx, nt, na) for nx in (1, 2, 3, 5, 7, 16, 31, 32, 33, 70) for nt in (1, 2, 9, 40) for na in (1, 2, 6, 7, 8, 15, 256, 300)]
    thin = [(1, 1, 60000), (2, 1, 20000), (3, 3, 8000), (3, 8000, 30), (5, 200, 200), (1, 200, 200)]
    text = "\n".join("%d %d %d" % s for s in shapes + thin)
    r = subprocess.run([exe], input=text, capture_output=True, text=True, check=True)
    rows = [tuple(map(int, line.split())) for line in r.stdout.splitlines()]
    assert len(rows) == len(shapes) + len(thin)
    assert not [s for s, (bad, ahead, _) in zip(shapes + thin, rows) if bad or ahead]
    # a thread per cell, an eighth more for the faces, and less than two for a column count that is no power of two
    for (nx, nt, na), (_, _, threads) in zip(thin, rows[len(shapes):]):
        assert threads < 2 * 8 / 7 * 1.05 * nx * nt * na, (nx, nt, na)
