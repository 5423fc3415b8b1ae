"""The scaled corner-vector forms of mahyco_amd/csrc/mh_geom.h on the host: cqs_hex_each,
cqs_hex_corner<L> and hex_volume give the bits of cqs_hex and cell_volume<8>, on the cells of
test_geom_host."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from tests.test_geom_host import HERE, _cells


def test_scaled_forms_equal_cqs_hex_bitwise(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "geom_forms_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off",
                    os.path.join(HERE, "host", "geom_forms_check.cpp"), "-o", exe], check=True)
    x = _cells(np.random.default_rng(7))
    words = np.ascontiguousarray(x).reshape(-1).view(np.uint64)
    text = "\n".join(" ".join(f"{w:x}" for w in words[i:i + 24]) for i in range(0, len(words), 24))
    r = subprocess.run([exe], input=text, capture_output=True, text=True, check=True)
    assert tuple(map(int, r.stdout.split())) == (len(x), 0)
