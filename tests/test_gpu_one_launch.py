"""The one-launch second-order pass (a tile forms the gradients it needs itself) against the oracle,
bit for bit, over the tile shapes at which its local cells, rounds of faces and launch shape change:
tiles of a few cells, tiles with more faces than two per thread, a single tile, more tiles than
compute units, blocks wider than the tile, and a scattered cell order whose neighbourhoods do not
fit in LDS (the two-pass form runs)."""
import numpy as np
import pytest

from cfd_solver_withcuda_amd import meshgen
from cfd_solver_withcuda_amd.solver import Mesh, Solver, cons_from_prim, make_config
from oracle.oracle import Oracle, make_cfg

pytestmark = pytest.mark.gpu

BCS = ("freestream", "exit", "wall", "wall", "wall")
FS = (1.4, 1.65, 0.0, 1.0)
# mesh (nx, ny), tile, face budget, renumber, block
SHAPES = [((40, 20), 128, 256, 1, 128), ((40, 20), 128, 256, 1, 256), ((50, 30), 256, 0, 1, 256),
          ((40, 20), 64, 0, 1, 64), ((120, 60), 16, 0, 1, 64), ((9, 5), 256, 0, 1, 256),
          ((120, 60), 128, 192, 1, 128), ((60, 40), 128, 0, 0, 128)]
SCHEMES = {
    "wlsq_rk3_lts": dict(flux="hllc", limiter="vanleer", gradient="wlsq", rk=3, lts=1),
    "gg_rk4": dict(flux="roe", limiter="minmod", gradient="gg", rk=4, lts=0),
    "wlsq_rk4_fallback": dict(flux="hllc", limiter="vanleer", gradient="wlsq", rk=4, lts=0, positivity=1),
    "gg_rk3_fallback": dict(flux="ausm", limiter="vanalbada", gradient="gg", rk=3, lts=0, positivity=2),
    "viscous": dict(flux="hllc", limiter="vanleer", gradient="wlsq", rk=3, lts=1, viscous="constant", mu=2e-3,
                    r_gas=1.0),
}


@pytest.fixture(scope="module")
def orc():
    return Oracle()


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s[0])) + "_" + "_".join(map(str, s[1:])))
@pytest.mark.parametrize("scheme", sorted(SCHEMES))
def test_steps_and_residual_vs_oracle(orc, shape, scheme):
    (nx, ny), tile, budget, renumber, block = shape
    print(f"case {shape} {scheme}", flush=True)
    m = meshgen.bump_mesh(nx, ny, 0.1, seed=17)
    cells = m.cells
    if not renumber:  # a scattered order
        cells = np.ascontiguousarray(cells[np.random.default_rng(3).permutation(len(cells))])
    om = orc.mesh(m.points, cells)
    ctr = om.arrays().ctr[: om.nphys]
    x, y = ctr[:, 0], ctr[:, 1]
    jump = np.where(x + 0.3 * y > 0.4, 1.0, 0.0)  # a front, so that the fallback has cells to redo
    U = cons_from_prim(1.4 * (1 + 0.1 * np.sin(3 * x) * np.cos(2 * y) + 0.8 * jump), 1.65 - 1.0 * jump,
                       0.1 * np.sin(2 * x), 1.0 + 0.1 * np.cos(5 * x + y) + 2.0 * jump)
    kw = dict(SCHEMES[scheme], order=2, roe_bdiss=1, cfl=0.6, bc=BCS, fs=FS)
    rk, lts = kw.pop("rk"), kw.pop("lts")
    s = Solver(Mesh(m.points, cells, tile=tile, face_budget=budget, renumber=renumber),
               make_config(rk=rk, lts=lts, block=block, grad_lds=0, **kw))
    s.set_state(U)
    ocfg = make_cfg(**kw)
    Ro, dto, go = om.residual(ocfg, U)
    R, dt, g = s.residual()
    assert np.array_equal(R, Ro) and np.array_equal(dt, dto) and np.array_equal(g, go)
    Uo, err_o = np.ascontiguousarray(U.copy()), []
    redone = 0
    for _ in range(3):
        err_o.append(om.step(ocfg, Uo, rk=rk, lts=lts)[0])
        redone += orc.last_fallback_cells()
    err, _ = s.step(3, history=True)
    assert np.array_equal(s.get_state(), Uo)
    # the error sums: the device adds tile by tile, the oracle cell by cell
    np.testing.assert_allclose(err, np.array(err_o), rtol=1e-12)
    if scheme == "wlsq_rk4_fallback" and nx >= 40:
        assert redone > 0
