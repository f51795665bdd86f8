"""States and residuals in the caller's cell order: around the ordering kernel's workgroups (256 values),
rows growing from call to call, several threads on one solver, and a batch, against the oracle and
against what was set."""
import threading

import numpy as np
import pytest

from cfd_solver_withcuda_amd import meshgen
from cfd_solver_withcuda_amd.batch import Batch
from cfd_solver_withcuda_amd.solver import Mesh, Solver, cons_from_prim, make_config
from oracle.oracle import Oracle, make_cfg

pytestmark = pytest.mark.gpu
KW = dict(flux="hllc", order=2, limiter="vanleer", gradient="wlsq", cfl=0.7, fs=(1.4, 1.65, 0.0, 1.0),
          bc=("freestream", "exit", "wall", "wall", "wall"))


def random_state(n, seed):
    r = np.random.default_rng(seed)
    return cons_from_prim(r.uniform(1.0, 1.5, n), r.uniform(1.2, 1.8, n), r.uniform(-0.2, 0.2, n), r.uniform(0.8, 1.2, n))


# cells x 4 values: 252, 256, 260 and more than one workgroup for one value per cell
@pytest.mark.parametrize("nx,ny", [(9, 7), (8, 8), (13, 5), (37, 7), (60, 31)])
def test_rows_vs_oracle(nx, ny):
    print(f"case rows {nx} x {ny}", flush=True)
    m = meshgen.bump_mesh(nx, ny, 0.08, seed=1, tri_frac=0.3)
    om = Oracle().mesh(m.points, m.cells)
    U = random_state(om.nphys, nx)
    s = Solver(Mesh(m.points, m.cells, tile=64), make_config(**KW))
    s.set_state(U)
    assert np.array_equal(s.get_state(), U)  # four values a cell, then eight
    Ro, dto, go = om.residual(make_cfg(**KW), U)
    R, dt, g = s.residual()
    assert np.array_equal(R, Ro) and np.array_equal(dt, dto) and np.array_equal(g, go)
    got = [None] * 4
    def get(i):
        got[i] = s.get_state()
    ts = [threading.Thread(target=get, args=(i,)) for i in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert all(np.array_equal(x, U) for x in got)


def test_batch_rows():
    print("case batch rows", flush=True)
    ms = [meshgen.bump_mesh(nx, 9, 0.08, seed=1) for nx in (7, 20, 33)]
    kw = {k: v for k, v in KW.items() if k != "fs"}
    b = Batch(ms, np.array([KW["fs"]] * 3), make_config(**kw, rk=3, lts=1))
    U = [random_state(len(m.cells), i) for i, m in enumerate(ms)]
    b.set_state(U)
    for _ in range(2):
        assert all(np.array_equal(x, u) for x, u in zip(b.get_state(), U))
