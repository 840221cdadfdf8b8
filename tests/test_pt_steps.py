"""Parallel-tempering steps decided by sa_ladder_exchange_steps: the driver asks for at most the
128 steps between two waits at a time (so its memory does not grow with the steps asked for), and
where the call has no memory, before any step or after some, the rest are stepped by the host with
the same draws, masks, energies and rates.  A model of the C ABI stands in for the device."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    exe = str(tmp_path_factory.mktemp("pt") / "pt_steps")
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Wno-unknown-pragmas", "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "dropin", "pt_steps.cpp"), "-o", exe], check=True)

    def run(mode, counts):
        r = subprocess.run([exe, mode, *map(str, counts)], capture_output=True, text=True, check=True)
        return r.stdout, r.stderr.strip()

    return run


@pytest.mark.parametrize("counts", [[1], [127, 2], [1000], [5, 128, 129, 3]])
def test_same_steps_with_and_without_memory(program, counts):
    out, most = program("device", counts)
    assert out.count("step ") == sum(counts)
    assert int(most) <= 128
    for mode in ("host", "breaks"):
        other, msg = program(mode, counts)
        assert other == out, mode
        assert "rror" not in msg
