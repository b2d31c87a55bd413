"""Memory that runs out in an FP64 pass, on a stand-in for the HIP runtime (fake_hip.cpp; no GPU): the
element scratch, the operator and its inverse blocks are needed, the tangents of the bricks only make the
CG faster, so a context without memory for those keeps passing and solves on the assembled operator."""

import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def fake_hip(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "libfakehip.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", so, os.path.join(HERE, "fake_hip.cpp")], check=True)
    return so


def test_an_fp64_pass_needs_no_memory_for_the_bricks(fake_hip):
    r = subprocess.run([sys.executable, os.path.join(HERE, "fake_hip_passes.py"), fake_hip, "5"], capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    runs = {f: rest for f, *rest in (tuple(int(w) for w in ln.split()) for ln in r.stdout.splitlines())}
    assert runs[-1] == [4, 0, 0, 1]  # four allocations, and the bricks
    for k in range(3):               # scratch, operator, inverse blocks
        assert runs[k][1] < 0
    assert runs[3] == [4, 0, 0, 0]   # the bricks' tangents: assembled
    assert runs[4] == [4, 0, 0, 1]   # none fails
