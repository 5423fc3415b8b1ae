"""The host side of the pinned read-back (mahyco_amd/csrc/mh_readback.h) on the CPU, over stand-ins of
the HIP calls (tests/host/hip_stub)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("readback") / "readback_check")
    subprocess.run(["g++", "-O2", "-g", "-std=c++17", "-pthread", "-I", os.path.join(HERE, "host", "hip_stub"),
                    os.path.join(HERE, "host", "readback_check.cpp"), "-o", exe], check=True)
    return exe


def _run(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    return tuple(map(int, r.stdout.split()))


def test_threads_share_the_slots(program):
    """Reads by several threads: each gets its own field, whatever the others read."""
    assert _run(program, "threads") == (48, 0)


def test_what_reads_pin(program):
    """A single read pins no more than it gains; pinned memory is bounded and given back."""
    assert _run(program, "pinning") == (66, 0)


def test_pinned_memory_is_short(program):
    """Where pinned memory is not to be had, or not enough, the field is read all the same."""
    assert _run(program, "short") == (9, 0)


def test_thread_of_another_device(program):
    """A case is read by threads whose current device is another than the case's (a new thread's is 0)."""
    assert _run(program, "device") == (4, 0)
