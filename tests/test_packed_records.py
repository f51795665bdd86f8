"""The records that meshes and batches copy to the device, by value against the layout, built with g++ under
AddressSanitizer and UndefinedBehaviorSanitizer. CPU only; skipped where g++ lacks the sanitizers."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from cfd_solver_withcuda_amd import meshgen

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_records_by_value(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not found")
    exe = str(tmp_path / "pack_checks")
    r = subprocess.run([gxx, "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined",
                        os.path.join(ROOT, "tests", "host", "pack_checks.cpp"),
                        os.path.join(ROOT, "cfd_solver_withcuda_amd", "csrc", "mesh_host.cpp"), "-o", exe],
                       capture_output=True, text=True)
    if r.returncode != 0 and ("sanitize" in r.stderr or "asan" in r.stderr):
        pytest.skip("g++ without sanitizer runtimes")
    assert r.returncode == 0, r.stderr
    paths = []
    for i, m in enumerate([meshgen.bump_mesh(60, 31, 0.1, seed=3, tri_frac=0.3), meshgen.shock_tube_mesh(5, 1)]):
        paths.append(str(tmp_path / f"m{i}.bin"))
        with open(paths[-1], "wb") as f:
            f.write(np.array([len(m.points), len(m.cells)], np.int32).tobytes())
            f.write(np.ascontiguousarray(m.points, np.float64).tobytes())
            f.write(np.ascontiguousarray(m.cells, np.int32).tobytes())
    r = subprocess.run([exe] + paths, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.count("checked") == 2, r.stdout + r.stderr
