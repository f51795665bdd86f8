"""States and residuals in the caller's cell order on either side of the size up to which the host orders
them (12288 cells): the oracle's values, each output asked for alone and together, on a stream of the
caller's, and a batch."""
import numpy as np
import pytest
import torch

from cfd_solver_withcuda_amd import meshgen
from cfd_solver_withcuda_amd._lib import check, dptr, lib
from cfd_solver_withcuda_amd.batch import Batch
from cfd_solver_withcuda_amd.solver import Mesh, Solver, cons_from_prim, make_config
from oracle.oracle import Oracle, make_cfg

pytestmark = pytest.mark.gpu
KW = dict(flux="hllc", order=2, limiter="vanleer", gradient="wlsq", cfl=0.7, fs=(1.4, 1.65, 0.0, 1.0),
          bc=("freestream", "exit", "wall", "wall", "wall"))


def random_state(n, seed):
    r = np.random.default_rng(seed)
    return cons_from_prim(r.uniform(1.0, 1.5, n), r.uniform(1.2, 1.8, n), r.uniform(-0.2, 0.2, n), r.uniform(0.8, 1.2, n))


@pytest.mark.parametrize("nx,ny", [(3, 2), (4095, 3), (128, 96), (4097, 3)])  # 6, 12285, 12288 and 12291 cells
@pytest.mark.parametrize("order", [1, 2])
def test_outputs_vs_oracle(nx, ny, order):
    print(f"case rows {nx} x {ny} order {order}", flush=True)
    m = meshgen.shock_tube_mesh(nx, ny)
    om = Oracle().mesh(m.points, m.cells)
    n = om.nphys
    assert n == nx * ny
    kw = dict(KW, order=order)
    U = random_state(n, nx)
    s = Solver(Mesh(m.points, m.cells, tile=128), make_config(block=128, **kw))
    s.set_state(U)
    assert np.array_equal(s.get_state(), U)
    want = om.residual(make_cfg(**kw), U)
    st = torch.cuda.Stream()
    for asked in ((1, 1, 1), (1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 0), (0, 0, 0)):
        out = [np.full((n, 4), np.nan), np.full(n, np.nan), np.full((n, 8), np.nan)]
        check(lib().cfd_residual(s.h, *[dptr(o) if a else None for o, a in zip(out, asked)], st.cuda_stream), "residual")
        for k in range(3 if order == 2 else 2):
            assert np.array_equal(out[k], want[k]) if asked[k] else np.isnan(out[k]).all(), (asked, k)


@pytest.mark.parametrize("sizes", [(5, 40), (120, 300, 945), (120, 300, 946)])  # 405, 12285 and 12294 cells
def test_batch_states(sizes):
    print(f"case batch rows {sizes}", flush=True)
    ms = [meshgen.shock_tube_mesh(nx, 9) for nx in sizes]
    kw = {k: v for k, v in KW.items() if k != "fs"}
    b = Batch(ms, np.array([KW["fs"]] * len(ms)), make_config(**kw, rk=3, lts=1))
    U = [random_state(len(m.cells), i) for i, m in enumerate(ms)]
    b.set_state(U)
    for _ in range(2):
        assert all(np.array_equal(x, u) for x, u in zip(b.get_state(), U))
