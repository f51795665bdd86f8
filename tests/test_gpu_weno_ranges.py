"""WENO face values outside the range where the weights' quotients go without range handling (values
above 2^200, a NaN in a line), at its edges (1e60) and for tiny and vanishing transverse momentum,
against the oracle's residual, bit for bit."""
import numpy as np
import pytest

from cfd_solver_withcuda_amd import meshgen
from cfd_solver_withcuda_amd.solver import Mesh, Solver, cons_from_prim, make_config
from oracle.oracle import Oracle, make_cfg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flux", ["hllc", "roe"])
@pytest.mark.parametrize("form", ["1e-30", "1e5", "1e60", "1e70", "tiny", "zero", "nan"])
def test_weno_residual_ranges_vs_oracle(flux, form):
    print(f"case weno range {form} {flux}", flush=True)
    m = meshgen.shock_tube_mesh(40, 20, length=2.0, height=1.0)
    om = Oracle().mesh(m.points, m.cells)
    x, y = om.arrays().ctr[:om.nphys].T[:2]
    r = np.random.default_rng(3)
    v = {"tiny": 1e-300 * r.uniform(-1, 1, len(x)), "zero": np.where(x < 1, 0.0, -0.0)}.get(form, 0.1 * np.sin(2 * x))
    U = cons_from_prim(1.4 + 0.2 * np.sin(3 * x) * np.cos(2 * y), 1.65 + 0.1 * np.cos(4 * y), v, np.where(x < 0.7, 2.0, 1.0))
    if form == "tiny":
        U[:, 2] = v  # not through the primitives: as small as it is
    if form[0] == "1":
        U[x > 0.4] *= float(form)
    if form == "nan":
        U[len(x) // 2 + 10, 3] = np.nan
    kw = dict(flux=flux, order=3, limiter="vanleer", gradient="wlsq", cfl=0.7,
              bc=("freestream", "exit", "wall", "wall", "wall"), fs=(1.4, 1.65, 0.0, 1.0))
    want, dto, _ = om.residual(make_cfg(**kw), U)
    s = Solver(Mesh(m.points, m.cells, tile=64), make_config(**kw))
    s.set_state(U)
    R, dt, _ = s.residual()
    fin = np.isfinite(want)
    assert np.array_equal(fin, np.isfinite(R)) and fin.mean() > 0.95
    assert np.array_equal(R[fin], want[fin]) and np.array_equal(dt, dto, equal_nan=True)
