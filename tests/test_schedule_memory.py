"""Host memory running out while a schedule is built, in any of the worker
threads, is an error code (a C++ program over the library's host source whose
allocations fail in turn)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from tycho2_amd import mesh as meshmod
from tycho2_amd.quadrature import product_quadrature
from tycho2_amd.sweeper import mesh_geometry

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "tycho2_amd", "csrc")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_failing_allocations_are_errors(tmp_path):
    sm = meshmod.kuhn_cube(4, 0.15, seed=7)
    conn = meshmod.tycho_connectivity(sm)
    omega, _ = product_quadrature(6)          # angles at 45 degrees
    _, area, normal = mesh_geometry(sm, conn)
    arrays = tmp_path / "mesh.bin"
    with open(arrays, "wb") as f:
        for a, t in (([sm.n_cells, len(omega)], np.int64),
                     (conn.adj_cell, np.int64), (area, np.float64),
                     (normal, np.float64), (omega, np.float64)):
            f.write(np.ascontiguousarray(a, dtype=t).tobytes())
    exe = tmp_path / "schedule_memory"
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off",
                    f"-I{INCLUDE}", f"-I{CSRC}",
                    os.path.join(HERE, "schedule_memory.cpp"),
                    os.path.join(CSRC, "t2_host.cpp"), "-o", str(exe),
                    "-lpthread"], check=True)
    res = subprocess.run([str(exe), str(arrays)], capture_output=True,
                         text=True, timeout=100)
    assert res.returncode == 0, res.stdout + res.stderr
    assert int(res.stdout.split()[-1]) > 50
