"""The reference iteration at the edges of its launches: time-step minima taken by the updates (up to
1024 partials) and by a launch of their own, residuals of fewer and of more tiles than compute units,
with and without the error's sums, against the oracle's steps, bit for bit."""
import numpy as np
import pytest

from cfd_solver_withcuda_amd import meshgen
from cfd_solver_withcuda_amd.solver import Mesh, Solver, make_config
from oracle.oracle import Oracle, make_cfg

pytestmark = pytest.mark.gpu
FS = (1.0, 0.0, 0.0, 1.0)


def sod_state(ctr):
    U = np.zeros((len(ctr), 4))
    left = ctr[:, 0] < 0.5
    U[:, 0] = np.where(left, 1.0, 0.125)
    U[:, 3] = np.where(left, 1.0, 0.1) / 0.4
    return U


# nx x ny cells in tiles of `tile`: 1, 250, 258, 516 and 1032 tiles
@pytest.mark.parametrize("nx,ny,tile", [(12, 5, 64), (320, 100, 128), (330, 100, 128), (330, 100, 64), (330, 100, 32)])
@pytest.mark.parametrize("rk,lts", [(3, 0), (3, 1), (1, 0)])
def test_reference_steps_vs_oracle(nx, ny, tile, rk, lts):
    print(f"case {nx} x {ny} tile {tile} rk {rk} lts {lts}", flush=True)
    m = meshgen.shock_tube_mesh(nx, ny)
    om = Oracle().mesh(m.points, m.cells)
    U0 = sod_state(om.arrays().ctr[:om.nphys])
    cfg = make_cfg(flux="roe", order=1, cfl=0.5, fs=FS)
    want = np.ascontiguousarray(U0.copy())
    for _ in range(3):
        om.step(cfg, want, rk=rk, lts=lts, ref=True)
    s = Solver(Mesh(m.points, m.cells, tile=tile), make_config(flux="roe", order=1, cfl=0.5, fs=FS, rk=rk, lts=lts, ref_mode=1))
    s.set_state(U0)
    s.step(3)
    assert np.array_equal(s.get_state(), want)
    s.set_state(U0)
    err, dt = s.step(3, history=True)
    assert np.array_equal(s.get_state(), want) and np.all(dt > 0.0)
    s.set_state(U0)
    _, steps, e = s.run_steady(0.0, 3, 3)
    assert steps == 3 and np.array_equal(e, err[-1]) and np.array_equal(s.get_state(), want)
