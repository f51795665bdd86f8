"""The tiles' neighbourhoods that the one-launch second-order pass indexes its local cells with,
built with g++ under AddressSanitizer and UndefinedBehaviorSanitizer and compared with the global
connectivity on generated meshes. CPU only; skipped where g++ lacks the sanitizers."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from cfd_solver_withcuda_amd import meshgen

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "host", "ring_checks.cpp")
MESH_HOST = os.path.join(ROOT, "cfd_solver_withcuda_amd", "csrc", "mesh_host.cpp")


def test_tile_rings_under_sanitizers(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not found")
    exe = str(tmp_path / "ring_checks")
    r = subprocess.run([gxx, "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined",
                        "-fno-sanitize-recover=undefined", SRC, MESH_HOST, "-o", exe], capture_output=True, text=True)
    if r.returncode != 0 and ("sanitize" in r.stderr or "asan" in r.stderr):
        pytest.skip("g++ without sanitizer runtimes")
    assert r.returncode == 0, r.stderr
    paths = []
    for i, m in enumerate([meshgen.bump_mesh(60, 31, 0.1, seed=3), meshgen.ffs_mesh(1.0 / 40, seed=4),
                           meshgen.shock_tube_mesh(5, 1), meshgen.ramp_mesh(33, 17, 15.0, seed=5, tri_frac=1.0)]):
        paths.append(str(tmp_path / f"m{i}.bin"))
        with open(paths[-1], "wb") as f:
            f.write(np.array([len(m.points), len(m.cells)], np.int32).tobytes())
            f.write(np.ascontiguousarray(m.points, np.float64).tobytes())
            f.write(np.ascontiguousarray(m.cells, np.int32).tobytes())
    r = subprocess.run([exe] + paths, capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "runtime error" not in r.stderr and r.stdout.count("checked") == len(paths), r.stdout + r.stderr
