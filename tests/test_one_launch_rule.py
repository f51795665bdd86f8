"""Which form a second-order pass takes: one launch where the tiles' neighbourhoods are small beside
the tiles or the mesh fits the chip at once, two launches where the cells' own order scatters a tile
over the mesh (there the one launch took up to twice as long). The results are those of the oracle on
either side."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from cfd_solver_withcuda_amd import meshgen

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def ordered(nx, ny, order):
    m = meshgen.bump_mesh(nx, ny, 0.08, seed=1, tri_frac=0.3)
    cells = m.cells
    if order == "shuffled":
        cells = np.ascontiguousarray(cells[np.random.default_rng(3).permutation(len(cells))])
    return m.points, cells


@pytest.fixture(scope="module")
def form(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not found")
    tmp = tmp_path_factory.mktemp("form")
    exe = str(tmp / "form_checks")
    subprocess.run([gxx, "-std=c++17", "-O2", os.path.join(ROOT, "tests", "host", "form_checks.cpp"),
                    os.path.join(ROOT, "cfd_solver_withcuda_amd", "csrc", "mesh_host.cpp"), "-o", exe], check=True)

    def run(mesh, shapes):
        path = str(tmp / "m.bin")
        with open(path, "wb") as f:
            f.write(np.array([len(mesh[0]), len(mesh[1])], np.int32).tobytes())
            f.write(np.ascontiguousarray(mesh[0], np.float64).tobytes())
            f.write(np.ascontiguousarray(mesh[1], np.int32).tobytes())
        r = subprocess.run([exe, path] + [str(v) for s in shapes for v in s], capture_output=True, text=True, check=True)
        return [int(v) for v in r.stdout.split()]
    return run


SHAPES = [(16, 64), (32, 64), (64, 64), (128, 128), (192, 256), (256, 256)]


@pytest.mark.parametrize("order", ["rows", "shuffled"])
def test_tiles_of_neighbours_take_one_launch(form, order):
    """Cells renumbered by the library: every shape, whatever the caller's order."""
    assert form(ordered(700, 350, order), [(t, 1, b) for t, b in SHAPES]) == [1] * 6


@pytest.mark.parametrize("order,small,large", [("rows", [1, 1, 1, 1, 1, 0], [1, 1, 0, 0, 0, 0]),
                                               ("shuffled", [1, 1, 1, 0, 0, 0], [0] * 6)])
def test_scattered_tiles_take_two(form, order, small, large):
    """In the caller's order: one launch while the chip holds all workgroups (20k cells) or the
    compute units stay occupied, two launches where the ring outweighs the tile (318k cells)."""
    assert form(ordered(180, 90, order), [(t, 0, b) for t, b in SHAPES]) == small
    assert form(ordered(700, 350, order), [(t, 0, b) for t, b in SHAPES]) == large


@pytest.mark.gpu
@pytest.mark.parametrize("scheme", ["wlsq", "gg_fallback", "viscous"])
@pytest.mark.parametrize("nx,ny,tile,block", [(60, 30, 32, 64), (330, 165, 32, 64), (420, 210, 128, 128)])
def test_both_forms_vs_oracle(scheme, nx, ny, tile, block):
    """Shuffled cells in tiles of 32 on either side of the chip's size, and rows in tiles of 128 beyond."""
    from cfd_solver_withcuda_amd.solver import Mesh, Solver, cons_from_prim, make_config
    from oracle.oracle import Oracle, make_cfg

    print(f"case {scheme} {nx}x{ny} tile {tile}", flush=True)
    pts, cells = ordered(nx, ny, "shuffled" if tile == 32 else "rows")
    om = Oracle().mesh(pts, cells)
    x, y = om.arrays().ctr[: om.nphys, :2].T
    jump = np.where(x + 0.3 * y > 0.4, 1.0, 0.0)
    U = cons_from_prim(1.4 * (1 + 0.1 * np.sin(3 * x) + 0.8 * jump), 1.65 - jump, 0.1 * np.sin(2 * x),
                       1.0 + 0.1 * np.cos(5 * x + y) + 2.0 * jump)
    rk, lts = (4, 0) if scheme == "gg_fallback" else (3, 1)
    kw = dict(flux="hllc", order=2, limiter="vanleer", gradient="gg" if rk == 4 else "wlsq", roe_bdiss=1, cfl=0.6,
              bc=("freestream", "exit", "wall", "wall", "wall"), fs=(1.4, 1.65, 0.0, 1.0))
    kw.update({"gg_fallback": dict(positivity=1), "viscous": dict(viscous="constant", mu=2e-3, r_gas=1.0)}.get(scheme, {}))
    s = Solver(Mesh(pts, cells, tile=tile, renumber=0), make_config(rk=rk, lts=lts, block=block, grad_lds=0, **kw))
    s.set_state(U)
    Uo = np.ascontiguousarray(U.copy())
    Ro, dto, go = om.residual(make_cfg(**kw), Uo)
    R, dt, g = s.residual()
    assert np.array_equal(R, Ro) and np.array_equal(dt, dto) and np.array_equal(g, go)
    for _ in range(2):
        om.step(make_cfg(**kw), Uo, rk=rk, lts=lts)
    s.step(2)
    assert np.array_equal(s.get_state(), Uo)
