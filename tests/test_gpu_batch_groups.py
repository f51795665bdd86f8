"""Batches whose instances are packed and copied in groups (small ones together, up to 32768 cells): every
instance marches as the same mesh alone, bit for bit, with the arrays of each order and gradient, whatever
the number of threads."""
import numpy as np
import pytest

from cfd_solver_withcuda_amd import meshgen
from cfd_solver_withcuda_amd.batch import Batch
from cfd_solver_withcuda_amd.solver import Mesh, Solver, cons_from_prim, make_config

pytestmark = pytest.mark.gpu
FS = (1.4, 1.65, 0.0, 1.0)
KW = dict(flux="hllc", limiter="vanleer", cfl=0.6, rk=3, lts=1, bc=("freestream", "exit", "wall", "wall", "wall"))
SCHEMES = {"first": dict(order=1), "wlsq": dict(order=2, gradient="wlsq"), "gg": dict(order=2, gradient="gg"),
           "weno": dict(order=3), "fallback": dict(order=2, gradient="gg", rk=4, positivity=1)}
# a single one; several around a group's cells, and one after them; one larger than a group between small ones
SIZES = [[(9, 5)], [(40, 20), (128, 200), (16, 399)], [(40, 20), (128, 200), (16, 400), (9, 5)],
         [(9, 5), (250, 160), (12, 7), (30, 20)]]


@pytest.mark.parametrize("scheme", sorted(SCHEMES))
@pytest.mark.parametrize("sizes", SIZES, ids=lambda s: "_".join(f"{a}x{b}" for a, b in s))
@pytest.mark.parametrize("threads", [1, 3])
def test_instances_march_as_alone(scheme, sizes, threads):
    print(f"case {scheme} {sizes} threads {threads}", flush=True)
    kw = dict(KW, **SCHEMES[scheme])
    tri = 0.0 if scheme == "weno" else 0.3
    ms = [meshgen.bump_mesh(nx, ny, 0.08, seed=i, tri_frac=tri) for i, (nx, ny) in enumerate(sizes)]
    b = Batch(ms, np.array([FS] * len(ms)), make_config(block=128, grad_lds=0, **kw), nthreads=threads)
    U = []
    for i, m in enumerate(ms):
        r = np.random.default_rng(i)
        n = len(m.cells)
        U.append(cons_from_prim(r.uniform(1.2, 1.5, n), r.uniform(1.4, 1.8, n), r.uniform(-0.1, 0.1, n), r.uniform(0.9, 1.1, n)))
    b.set_state(U)
    b.solve(tol=-1.0, max_steps=2, check_every=2)
    got = b.get_state()
    for i, m in enumerate(ms):
        s = Solver(Mesh(m.points, m.cells, tile=128, face_budget=256), make_config(block=128, grad_lds=0, fs=FS, **kw))
        s.set_state(U[i])
        s.step(2)
        assert np.array_equal(got[i], s.get_state()), i
