"""Creating a device mesh where host memory runs out: an error, not an end of the process, wherever it
happens (the layout, the packed records, the neighbourhoods and their thread)."""
import subprocess
import sys

import pytest

CHILD = """
import ctypes, resource, sys
import numpy as np
from cfd_solver_withcuda_amd import meshgen
from cfd_solver_withcuda_amd._lib import dptr, iptr, lib
m = meshgen.shock_tube_mesh(400, 250)
L, p, h = lib(), ctypes.c_void_p(), ctypes.c_void_p()
L.cfd_device_alloc(16, ctypes.byref(p))  # the runtime is up (or has found no device) before the limit
pts, cells = np.ascontiguousarray(m.points), np.ascontiguousarray(m.cells, np.int32)
vm = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (vm + int(sys.argv[1]) * 2 ** 20,) * 2)
rc = L.cfd_mesh_create(len(pts), dptr(pts), len(cells), iptr(cells), 128, 0, 1, ctypes.byref(h))
print("rc", rc)
"""


@pytest.mark.parametrize("first", [40, 60, 80, 100])
def test_out_of_memory_is_an_error(first):
    """100k cells take about 85 MB on the host."""
    ends = []
    for mb in range(first, first + 20, 4):
        r = subprocess.run([sys.executable, "-c", CHILD, str(mb)], capture_output=True, text=True, timeout=120)
        ends.append((mb, r.returncode, r.stdout.strip() or r.stderr[-200:]))
    print(ends)
    assert all(rc == 0 and out.startswith("rc ") for _, rc, out in ends), ends
