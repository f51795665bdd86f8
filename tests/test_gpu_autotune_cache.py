"""The autotune cache's keys: an entry is used only for the kernels that it was timed with, and for the
scheme options that select other kernels."""
import json

import numpy as np
import pytest

from cfd_solver_withcuda_amd import build, meshgen
from cfd_solver_withcuda_amd.batch import Batch
from cfd_solver_withcuda_amd.solver import make_config

KW = dict(flux="hllc", order=2, limiter="vanleer", gradient="wlsq", cfl=0.7, rk=3, lts=1, block=0,
          bc=("freestream", "exit", "wall", "wall", "wall"))


def source(**kw):
    ms = [meshgen.bump_mesh(20, 9, 0.08, seed=1), meshgen.bump_mesh(30, 9, 0.08, seed=2)]
    i = Batch(ms, np.array([(1.4, 1.65, 0.0, 1.0)] * 2), make_config(**dict(KW, **kw))).info()
    return i["shape_source"], (i["tile"], i["face_budget"], i["block"])


@pytest.mark.gpu
def test_entries_of_other_kernels_and_options_are_not_used(tmp_path, monkeypatch):
    path = tmp_path / "autotune.json"
    monkeypatch.setenv("CFD_AUTOTUNE_CACHE", str(path))
    print("case autotune cache", flush=True)
    assert source()[0] == "autotuned"
    (key,) = json.loads(path.read_text())
    # the same batch as earlier kernels left it: keys without the kernels and options, or another digest
    old = [key.split("|pos")[0], key[:-4] + ("0000" if key[-4:] != "0000" else "1111")]
    path.write_text("{\n" + ",\n".join(f'"{k}": [64, 96, 64, 1e-9]' for k in old) + "\n}\n")
    src, shape = source()
    assert src == "autotuned" and shape != (64, 96, 64)
    assert source()[0] == "autotune cache"
    # the fallback and limiter freezing run other kernels
    assert source(positivity=1)[0] == "autotuned"
    assert source(freeze_stall=300)[0] == "autotuned"
    assert len(json.loads(path.read_text())) == 5


def test_the_digest_follows_sources_and_options(tmp_path, monkeypatch):
    (tmp_path / "fv_a.hip").write_text("one")
    (tmp_path / "mlp_a.hip").write_text("one")
    monkeypatch.setattr(build, "CSRC", str(tmp_path))
    d = build.kernel_digest()
    assert d == build.kernel_digest() and d != build.kernel_digest(("CFD_FLUX_WAVES_PER_EU=4",))
    (tmp_path / "mlp_a.hip").write_text("two")
    assert build.kernel_digest() == d
    (tmp_path / "fv_a.hip").write_text("two")
    assert build.kernel_digest() != d
