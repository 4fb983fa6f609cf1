"""What the library's calls leave running on their streams, with a HIP runtime of the host alone
(tests/host/hip_stub.cpp): no launch is under way when a step has returned, failed or not -- the
next step's first launches are ordered after the main stream only."""
from __future__ import annotations

import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(os.path.dirname(HERE), "sdfibm_amd", "libsdfibm_hip.so")

SCRIPT = """
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
stub.stub_busy.restype = ctypes.c_longlong
import numpy as np
from sdfibm_amd import mesh as M, solids as S
from sdfibm_amd._lib import SdfibmError
from sdfibm_amd.cloud import SolidCloud
m = M.uniform_box((100, 90, 80), (0, 0, 0), (100.0, 90.0, 80.0))
sol = S.make_solids(4)
sol["shape"][3] = S.PLANE
sol["prm"][:3, 0] = 3.0, 8.0, 36.0  # small, medium and big tiles
sol["center"] = [(9, 9, 9), (30, 20, 20), (50, 45, 40), (50, 4.3, 40)]
c = SolidCloud(m, precision="fp32")
c.set_solids(sol)
for fail in (0, 1, 0):
    sol["center"][3, 1] += 1.0  # the plane is labelled again
    c.set_solids(sol)
    stub.stub_fail_copies(fail)
    try:
        c.interact(0.0, 1e-3)
        failed = 0
    except SdfibmError:
        failed = 1
    print("failed", failed, "asked", fail, "busy", stub.stub_busy(), flush=True)
"""


@pytest.mark.skipif(not os.path.exists(LIB), reason="library not built")
def test_a_failed_step_leaves_nothing_running(tmp_path):
    stub = str(tmp_path / "hip_stub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-w", "-o", stub,
                    os.path.join(HERE, "host", "hip_stub.cpp")], check=True, timeout=120)
    env = dict(os.environ, PYTHONPATH=os.path.dirname(HERE))
    r = subprocess.run([sys.executable, "-c", SCRIPT, stub], capture_output=True, text=True, timeout=120, env=env)
    assert r.returncode == 0, r.stderr
    assert r.stdout.split("\n")[:3] == [f"failed {f} asked {f} busy 0" for f in (0, 1, 0)], r.stdout
