"""The cell bins of general meshes, with a HIP runtime of the host alone (tests/host/hip_stub.cpp): about
one bin per four cells whatever the mesh's proportions -- a mesh one cell thick, whose cell centres
lie in a plane up to rounding, thin slabs, a single row of cells."""
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
stub.stub_bytes.restype = ctypes.c_longlong
from sdfibm_amd import mesh as M
from sdfibm_amd.cloud import SolidCloud
for n, h in (((106, 112, 1), (0.711, 0.711, 0.711)), ((90, 120, 2), (1.0, 1.0, 1e-4)), ((70, 1, 90), (0.3, 0.7, 0.3)),
             ((4000, 1, 1), (0.1, 0.1, 0.1)), ((30, 28, 26), (1.0, 1.0, 1.0))):
    lo = [-0.5 * a * b for a, b in zip(n, h)]
    pm = M.uniform_box(n, lo, [-a for a in lo]).to_polymesh()
    before = stub.stub_bytes()
    SolidCloud(pm, two_d=n[2] == 1, precision="fp32").close()
    print((stub.stub_bytes() - before) // pm.n_cells, flush=True)
"""


@pytest.mark.skipif(not os.path.exists(LIB), reason="library not built")
def test_bins_are_as_many_as_the_cells_ask_for(tmp_path):
    stub = str(tmp_path / "hip_stub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-w", "-o", stub,
                    os.path.join(HERE, "host", "hip_stub.cpp")], check=True, timeout=120)
    env = dict(os.environ, PYTHONPATH=os.path.dirname(HERE))
    r = subprocess.run([sys.executable, "-c", SCRIPT, stub], capture_output=True, text=True, timeout=120, env=env)
    assert r.returncode == 0, r.stderr
    per_cell = [int(v) for v in r.stdout.split()]
    # a hexahedral cell's points, faces, lists, fields and share of a bin: about 400 to 600 bytes
    assert len(per_cell) == 5 and all(v < 1000 for v in per_cell), per_cell
