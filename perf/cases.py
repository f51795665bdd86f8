"""Performance cases of the framework: the work its users have it do, through its entry points.

`listed()` gives the standing cases and `draw(rng)` further ones of the same ranges; `prepare` makes
what a program has in hand before a call, `run` is one pass of it, `work` the bytes and operations a
pass cannot do without, and `exact` its results by plain torch in 64 bits.

Kinds of case:
  march       time steps of one solver (`Solver.step`, or `Solver.run_steady` for a steady march)
  residual    `Solver.residual`: net flux, local time step and gradients into host arrays
  batch       a batch of uneven ramps marched together (`Batch.solve`)
  wrappers    the reference-layout wrappers on caller-owned device arrays (`launch_*`)
  mlp_train   Adam steps of the warm start's coordinate network (`MLP.train`)
  mlp_predict its prediction on cell centres (`MLP.predict`)
"""
from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch

from cfd_solver_withcuda_amd import cases as families
from cfd_solver_withcuda_amd import meshgen
from cfd_solver_withcuda_amd._lib import check, lib
from cfd_solver_withcuda_amd.batch import Batch
from cfd_solver_withcuda_amd.solver import REF_BCS, Mesh, Solver, freestream, make_config
from cfd_solver_withcuda_amd.surrogate import MLP

DEV = "cuda"
F64 = torch.float64
GM1 = 1.4 - 1.0

# Tile and launch settings: "tuned" as bench.py has them, "doc" as the integration guide's example
# has them (128-cell tiles, the configuration's defaults), "plain" the library's defaults.
SHAPES = {
    "tuned": (dict(tile=128, face_budget=256), dict(block=128, grad_lds=0)),
    "doc": (dict(tile=128, face_budget=256), dict()),
    "plain": (dict(), dict()),
}


# ---- the cases -------------------------------------------------------------------------------


def _march(name, mesh, n, shape, nsteps, call="step", **scheme):
    return dict(name=name, kind="march", mesh=mesh, n=n, shape=shape, nsteps=nsteps, call=call, **scheme)


def _scheme(flux="hllc", order=2, limiter="vanleer", gradient="wlsq", rk=3, lts=1, ref_mode=0, positivity=0,
            viscous="off", cfl=0.8):
    return dict(flux=flux, order=order, limiter=limiter, gradient=gradient, rk=rk, lts=lts, ref_mode=ref_mode,
                positivity=positivity, viscous=viscous, cfl=cfl)


def listed():
    return [
        # the reference's own iteration on its shock-tube problem: a 16k-cell mesh, launch-bound
        _march("sod_reference", "sod", 40, "doc", 20,
               **_scheme("roe", 1, rk=3, lts=0, ref_mode=1, cfl=0.5)),
        # a steady march of a small mesh with the library's default tiles: the smallest calls
        _march("bump_small_steady", "bump", 31, "plain", 50, "steady", **_scheme()),
        # the 1.27M-cell channel bump, local time stepping: what a steady solve repeats
        _march("bump_march", "bump", 700, "tuned", 2, **_scheme()),
        # the 8M-cell forward step, Mach 3, RK4 with the positivity fallback: the headline workload
        _march("step_rk4", "ffs", 1560, "tuned", 1, **_scheme(rk=4, lts=0, positivity=1, cfl=0.4)),
        # the same geometry with Roe, minmod and Green-Gauss gradients, a middling mesh
        _march("step_roe_gg", "ffs", 521, "tuned", 2,
               **_scheme("roe", 2, "minmod", "gg", rk=4, lts=0, positivity=1, cfl=0.4)),
        # laminar flow over the bump, no-slip walls, as the integration guide sets it up
        _march("bump_viscous", "bump", 351, "doc", 3, **_scheme(viscous="constant")),
        # WENO5 on quadrilaterals
        _march("bump_weno", "bump", 450, "tuned", 2, **_scheme(order=3)),
        # a batch of uneven compression ramps, every other one from a warm start (frozen limiter)
        dict(name="ramp_batch", kind="batch", instances=16, min_cells=20000, max_cells=120000, nsteps=40),
        # net flux, time step and gradients handed back to a host program
        dict(name="residual_host", kind="residual", mesh="bump", n=151, shape="doc", **_scheme()),
        # a program written on the reference's per-cell wrappers: limiter, MUSCL, flux, RK3 stage
        dict(name="wrappers", kind="wrappers", n=600, flux="hllc"),
        # the warm start's network: training steps on 16k-row minibatches
        dict(name="mlp_train", kind="mlp_train", width=256, depth=6, batch=16384, samples=1 << 18, nsteps=10),
        # its prediction on a mesh's cell centres
        dict(name="mlp_predict", kind="mlp_predict", width=256, depth=6, rows=200003),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["march", "march", "march", "march", "march", "residual", "batch", "wrappers", "mlp_train",
                       "mlp_predict"])
    shape = rng.choice(sorted(SHAPES))
    if kind == "march":
        form = rng.choice(["euler", "euler", "fallback", "viscous", "weno", "reference"])
        call = "step"
        if form == "reference":
            s = _scheme(rng.choice(["roe", "llf"]), 1, rk=3, lts=0, ref_mode=1, cfl=0.5)
            return dict(kind=kind, mesh="sod", n=_log(rng, 10, 160), shape=shape, nsteps=rng.randint(5, 30), call=call, **s)
        if form == "euler":
            call = rng.choice(["step", "steady"])
            s = _scheme(rng.choice(["hllc", "roe", "ausm"]), rng.choice([1, 2, 2, 2]),
                        rng.choice(["vanleer", "minmod", "vanalbada"]), rng.choice(["wlsq", "wlsq", "gg"]))
            mesh, n = "bump", _log(rng, 20, 900)
        elif form == "fallback":
            s = _scheme(rng.choice(["hllc", "roe"]), 2, rng.choice(["vanleer", "minmod"]),
                        rng.choice(["wlsq", "gg"]), rk=rng.choice([3, 4]), lts=0, positivity=rng.choice([1, 1, 2]), cfl=0.4)
            mesh, n = "ffs", _log(rng, 30, 900)
        elif form == "viscous":
            s = _scheme(viscous="constant")
            mesh, n = "bump", _log(rng, 20, 600)
        else:
            s = _scheme(order=3)
            mesh, n = "bump", _log(rng, 20, 600)
        return dict(kind=kind, mesh=mesh, n=n, shape=shape, nsteps=rng.randint(1, 4), call=call, **s)
    if kind == "residual":
        return dict(kind=kind, mesh="bump", n=_log(rng, 20, 400), shape=shape,
                    **_scheme(rng.choice(["hllc", "roe"]), rng.choice([1, 2]), gradient=rng.choice(["wlsq", "gg"])))
    if kind == "batch":
        lo = _log(rng, 3000, 30000)
        return dict(kind=kind, instances=rng.randint(3, 24), min_cells=lo, max_cells=lo * rng.randint(2, 8),
                    nsteps=rng.randint(5, 40))
    if kind == "wrappers":
        return dict(kind=kind, n=_log(rng, 20, 1000), flux=rng.choice(["hllc", "roe", "llf"]))
    width, depth = rng.choice([(128, 4), (256, 6), (256, 6), (192, 5)])
    if kind == "mlp_train":
        return dict(kind=kind, width=width, depth=depth, batch=512 * rng.randint(2, 64),
                    samples=_log(rng, 20000, 1 << 19), nsteps=rng.randint(2, 12))
    return dict(kind=kind, width=width, depth=depth, rows=_log(rng, 500, 1000000))


# ---- meshes and states -----------------------------------------------------------------------


@functools.lru_cache(maxsize=None)
def _points_cells(mesh, n, quads):
    """Generated points and cells: `n` cells across the channel's height."""
    tri = 0.0 if quads else 0.3
    if mesh == "sod":
        m = meshgen.shock_tube_mesh(10 * n, n)
    elif mesh == "bump":
        m = meshgen.bump_mesh(2 * n, n, 0.08, seed=1, tri_frac=tri)
    else:
        m = meshgen.ffs_mesh(1.0 / n, seed=2, tri_frac=tri)
    return m.points, m.cells


def _quads(case):
    return case.get("order") == 3 or case["mesh"] == "sod"


@functools.lru_cache(maxsize=None)
def _mesh(mesh, n, quads, shape, device):
    """The mesh handle a program keeps (one for all its states), and the cell centres."""
    pts, cells = _points_cells(mesh, n, quads)
    return Mesh(pts, cells, device=device, **SHAPES[shape][0])


def _centres(pts, cells):
    c = torch.as_tensor(cells, device=DEV).long()
    ok = (c >= 0).to(F64)
    xy = torch.as_tensor(pts[:, :2], device=DEV, dtype=F64)[c.clamp(min=0)] * ok[:, :, None]
    return xy.sum(1) / ok.sum(1, keepdim=True)


def _flow(ctr, fs, seed):
    """A developing flow: the prescribed state with smooth disturbances of several wavelengths and
    two fronts in density and pressure, placed by the seed."""
    r = np.random.default_rng(seed)
    x, y = ctr[:, 0], ctr[:, 1]
    rho0, u0, v0, p0 = fs
    a = math.sqrt(1.4 * p0 / rho0)
    d = torch.zeros(4, len(x), dtype=F64, device=DEV)
    for k in (2.0, 5.0, 13.0, 29.0):
        for q in range(4):
            th, ph = r.uniform(0, 2 * math.pi, 2)
            d[q] += 0.04 / k ** 0.5 * torch.sin(k * (math.cos(th) * x + math.sin(th) * y) + ph)
    front = torch.zeros_like(x)
    for _ in range(2):
        th, at = r.uniform(-0.6, 0.6), r.uniform(0.2, 0.9)
        front += 0.15 * torch.tanh(80.0 * (x - at - math.tan(th) * (y - 0.5)))
    rho = rho0 * (1 + d[0] + 0.7 * front)
    p = p0 * (1 + d[3] + front)
    u = u0 + a * (d[1] - 0.2 * front)
    v = v0 + a * d[2]
    return torch.stack([rho, rho * u, rho * v, p / GM1 + 0.5 * rho * (u * u + v * v)], 1)


def _shock_tube(ctr, seed):
    r = np.random.default_rng(seed)
    at, rl, pl = 0.5 + r.uniform(-0.1, 0.1), 1.0 + r.uniform(-0.1, 0.1), 1.0 + r.uniform(-0.1, 0.1)
    left = ctr[:, 0] < at
    rho = torch.where(left, rl, 0.125 * torch.ones_like(ctr[:, 0]))
    p = torch.where(left, pl, 0.1 * torch.ones_like(ctr[:, 0]))
    z = torch.zeros_like(rho)
    return torch.stack([rho, z, z, p / GM1], 1)


def _flow_setup(case):
    """The scheme's keywords and prescribed state of a single-mesh case."""
    if case["mesh"] == "sod":
        fs, bc, bdiss = (1.0, 0.0, 0.0, 1.0), REF_BCS, 0
    else:
        fs, bc, bdiss = freestream(3.0 if case["mesh"] == "ffs" else 1.65), families.BUMP_BCS, 1
    kw = {k: case[k] for k in ("flux", "order", "limiter", "gradient", "rk", "lts", "ref_mode", "positivity", "cfl")
          if k in case}
    if case.get("viscous", "off") != "off":
        # Reynolds number 1e4 per unit length, no-slip lower wall and bump
        bc = ("freestream", "exit", "symmetry", "noslip_wall", "noslip_wall")
        kw.update(viscous=case["viscous"], mu=fs[0] * fs[1] / 1e4, prandtl=0.72, r_gas=1.0)
    fs = tuple(float(v) for v in fs)
    return dict(kw, bc=bc, fs=fs, roe_bdiss=bdiss)


def _state(case, seed):
    pts, cells = _points_cells(case["mesh"], case["n"], _quads(case))
    ctr = _centres(pts, cells)
    return _shock_tube(ctr, seed) if case["mesh"] == "sod" else _flow(ctr, _flow_setup(case)["fs"], seed)


class _View:
    """A device buffer of a solver as torch sees it (no copy); it keeps the solver alive, since
    the buffer is freed with it."""

    def __init__(self, solver, ptr, n):
        self.solver = solver
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=(n, 4), typestr="<f8", version=2)


# ---- prepare and run -------------------------------------------------------------------------


def prepare(case, seed):
    return globals()["_prepare_" + ("solver" if case["kind"] in ("march", "residual") else case["kind"])](case, seed)


def run(state):
    return globals()["_run_" + state["case"]["kind"]](state)


def _prepare_solver(case, seed):
    mesh = _mesh(case["mesh"], case["n"], _quads(case), case["shape"], True)
    s = Solver(mesh, make_config(**_flow_setup(case), **SHAPES[case["shape"]][1]))
    s.set_state(_state(case, seed).cpu().numpy())
    return dict(case=case, solver=s, views={})


def _run_march(state):
    case, s = state["case"], state["solver"]
    out = {}
    if case["call"] == "steady":
        _, out["steps"], out["error"] = s.run_steady(1e-8, case["nsteps"], case["nsteps"])
    else:
        s.step(case["nsteps"])
    ptr = s.state_device_ptr()  # the resident state, in the mesh's renumbered order
    if ptr not in state["views"]:
        state["views"][ptr] = torch.as_tensor(_View(s, ptr, s.mesh.nphys), device=DEV)
    out["U"] = state["views"][ptr]
    return out


def _run_residual(state):
    R, dt, grad = state["solver"].residual()
    return dict(R=R, dt=dt, grad=grad) if state["case"]["order"] > 1 else dict(R=R, dt=dt)


@functools.lru_cache(maxsize=None)
def _ramps(instances, min_cells, max_cells):
    return families.ramp_batch(instances, min_cells=min_cells, max_cells=max_cells)


def _batch_scheme():
    return dict(flux="ausm", order=2, limiter="vanleer", gradient="wlsq", cfl=1.2, rk=3, lts=1, roe_bdiss=1,
                bc=families.RAMP_BCS)


def _batch_states(case, seed):
    cs = _ramps(case["instances"], case["min_cells"], case["max_cells"])
    return [_flow(_centres(c.mesh.points, c.mesh.cells), tuple(float(v) for v in c.fs), 1000 * seed + i)
            for i, c in enumerate(cs)]


def _prepare_batch(case, seed):
    cs = _ramps(case["instances"], case["min_cells"], case["max_cells"])
    b = Batch([c.mesh for c in cs], np.array([c.fs for c in cs]),
              make_config(block=128, grad_lds=0, freeze_stall=300, **_batch_scheme()))
    b.set_state([u.cpu().numpy() for u in _batch_states(case, seed)])
    b.set_freeze([i % 2 for i in range(case["instances"])])
    return dict(case=case, batch=b)


def _run_batch(state):
    b, n = state["batch"], state["case"]["nsteps"]
    r = b.solve(1e-8, max_steps=n, check_every=n)
    return dict(U=b.get_state(), error0=r["err"][:, 0], steps=r["steps"], status=r["status"])


def _prepare_wrappers(case, seed):
    pts, cells = _points_cells("bump", case["n"], True)
    g = _Faces(pts, cells)
    U = _flow(g.ctr, tuple(float(v) for v in freestream(1.65)), seed)
    W = _prims(U)
    P6 = torch.stack([W[0], W[1], W[2], W[3], W[3] / (W[0] * 287.0), W[4]], 1).contiguous()
    t = g.per_cell()
    N = len(U)
    z = lambda: torch.zeros(N, 4, 4, dtype=F64, device=DEV)  # noqa: E731
    net = 1e-3 * U.roll(1, 0)
    return dict(case=case, N=N, U=U.contiguous(), P=P6, nb=t["nbr"].int().contiguous(), nrm=t["nrm"].contiguous(),
                len=t["len"].contiguous(), dist=t["dist"].contiguous(), net=net.contiguous(),
                ia=(1.0 / g.area).contiguous(), phi=z(), QL=z(), QR=z(), F=z(), Urk=torch.zeros_like(U))


def _run_wrappers(s):
    L, N, st = lib(), s["N"], ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    p = lambda k: ctypes.c_void_p(s[k].data_ptr())  # noqa: E731
    d = ctypes.c_double
    check(L.launch_vanleer_limiter(p("U"), p("nb"), p("dist"), p("phi"), N, d(0.5), 256, st), "launch_vanleer_limiter")
    check(L.launch_muscl_reconstruction(p("U"), p("nb"), p("dist"), p("phi"), p("QL"), p("QR"), N, d(0.5), 256, st),
          "launch_muscl_reconstruction")
    check(getattr(L, "launch_%s_flux" % s["case"]["flux"])(p("U"), p("P"), p("nb"), p("nrm"), p("len"), p("F"), N,
                                                          d(1.4), 256, st), "launch flux")
    check(L.launch_tvd_rk3_stage(p("U"), p("net"), None, p("Urk"), p("ia"), d(1e-5), N, 1, 256, st),
          "launch_tvd_rk3_stage")
    return {k: s[k] for k in ("phi", "QL", "QR", "F", "Urk")}


def _samples(n, seed):
    """Cell centres, Mach number and thickness, and the primitives of a bump-like flow there."""
    r = np.random.default_rng(seed)
    feat = np.column_stack([r.uniform(-1, 2, n), r.uniform(0, 1, n), r.uniform(1.2, 3.0, n),
                            r.uniform(0.04, 0.12, n)]).astype(np.float32)
    x, y, M, t = feat.T.astype(np.float64)
    shock = np.tanh(12.0 * (x - y * np.sqrt(M * M - 1.0)))
    targ = np.column_stack([1.4 * (1 + 2 * t * shock), M * (1 - t * shock), t * np.sin(3 * x) * (1 - y),
                            1 + 3 * t * shock]).astype(np.float32)
    return feat, targ


def _network(case, seed, max_rows):
    m = MLP(4, case["width"], case["depth"], 4, max_rows=max_rows, seed=seed % 1000)
    m.fit_normalization(*_samples(4096, seed + 1))
    return m


def _prepare_mlp_train(case, seed):
    feat, targ = _samples(case["samples"], seed)
    return dict(case=case, mlp=_network(case, seed, case["batch"]), feat=feat, targ=targ)


def _run_mlp_train(s):
    c = s["case"]
    hist = s["mlp"].train(s["feat"], s["targ"], c["nsteps"], batch=c["batch"], log_every=c["nsteps"])
    W, b = s["mlp"].get_params()
    return dict(W=W, b=b, loss=hist)


def _prepare_mlp_predict(case, seed):
    return dict(case=case, mlp=_network(case, seed, 65536), feat=_samples(case["rows"], seed)[0])


def _run_mlp_predict(s):
    return s["mlp"].predict(s["feat"])


# ---- work ------------------------------------------------------------------------------------


def work(case):
    """Bytes: each input read once and each output written once. A march of k steps reads its state
    and its mesh (per face two cells, normal, length and centre offset; per cell area) and writes
    its state; operations are per face and stage, with one division or root as one."""
    kind = case["kind"]
    if kind in ("march", "residual"):
        pts, cells = _points_cells(case["mesh"], case["n"], _quads(case))
        C = len(cells)
        F = int((cells >= 0).sum()) // 2
        mesh = 48 * F + 8 * C
        per_face = (250 if case["order"] == 2 else 700 if case["order"] == 3 else 120)
        if case.get("viscous", "off") != "off":
            per_face += 120
        if kind == "residual":
            return dict(bytes=mesh + C * (32 + 32 + 8 + (64 if case["order"] > 1 else 0)), flops=per_face * F)
        stages = (4 if case["rk"] == 4 else 3) * case["nsteps"]
        return dict(bytes=mesh + 64 * C, flops=stages * (per_face * F + 40 * C))
    if kind == "batch":
        cs = _ramps(case["instances"], case["min_cells"], case["max_cells"])
        C = sum(len(c.mesh.cells) for c in cs)
        F = sum(int((c.mesh.cells >= 0).sum()) // 2 for c in cs)
        return dict(bytes=48 * F + 72 * C, flops=3 * case["nsteps"] * (250 * F + 40 * C))
    if kind == "wrappers":
        N = 2 * case["n"] * case["n"]
        per = 32 + 48 + 16 + 64 + 32 + 32 + 32 + 8 + 4 * 128 + 32
        return dict(bytes=N * per, flops=N * 4 * 150)
    w, d = case["width"], case["depth"]
    nw = 4 * w + (d - 1) * w * w + 4 * w
    if kind == "mlp_train":
        return dict(bytes=32 * case["samples"] + 24 * nw, flops=6 * nw * case["batch"] * case["nsteps"])
    return dict(bytes=32 * case["rows"] + 4 * nw, flops=2 * nw * case["rows"])


# ---- exact: plain torch in 64 bits -----------------------------------------------------------


class _Faces:
    """Faces and geometry of a mixed mesh: per face its two cells (right = -1 on the boundary), the
    unit normal from the left cell, length, centre offset and boundary kind."""

    def __init__(self, pts, cells):
        P = torch.as_tensor(pts[:, :2], device=DEV, dtype=F64)
        C = torch.as_tensor(cells, device=DEV).long()
        self.nc = n = len(C)
        self.nf = nf = 3 + (C[:, 3] >= 0).long()
        self.ctr = _centres(pts, cells)
        f = torch.arange(4, device=DEV)
        valid = f[None] < nf[:, None]
        a = C.clamp(min=0)
        b = torch.gather(a, 1, (f[None] + 1) % nf[:, None])
        pa, pb = P[a], P[b]
        cross = (pa[..., 0] * pb[..., 1] - pb[..., 0] * pa[..., 1]) * valid
        self.area = 0.5 * cross.sum(1).abs()
        he_cell, he_slot = valid.nonzero(as_tuple=True)
        ha, hb = a[valid], b[valid]
        key = torch.minimum(ha, hb) * len(P) + torch.maximum(ha, hb)
        uk, face = torch.unique(key, return_inverse=True)
        m = len(uk)
        ids = torch.arange(len(key), device=DEV)
        first = torch.full((m,), len(key), device=DEV).scatter_reduce(0, face, ids, "amin")
        last = torch.zeros(m, dtype=torch.long, device=DEV).scatter_reduce(0, face, ids, "amax")
        self.L = he_cell[first]
        self.inner = first != last
        self.R = torch.where(self.inner, he_cell[last], -1)
        self.sL, self.sR = he_slot[first], he_slot[last]
        A, B = P[ha[first]], P[hb[first]]
        d = B - A
        self.dl = d.norm(dim=1)
        self.nx, self.ny = d[:, 1] / self.dl, -d[:, 0] / self.dl
        other = torch.where(self.inner[:, None], self.ctr[self.R.clamp(min=0)], A + B - self.ctr[self.L])
        self.d = other - self.ctr[self.L]
        lo, hi = P.min(0).values, P.max(0).values
        kind = torch.full((m,), 5, device=DEV)
        for k, q, edge in ((3, 1, hi), (4, 1, lo), (2, 0, hi), (1, 0, lo)):
            kind[((A[:, q] - edge[q]).abs() < 1e-6) & ((B[:, q] - edge[q]).abs() < 1e-6)] = k
        self.kind = kind
        self.face = torch.full((n, 4), -1, device=DEV)
        self.face[valid] = face

    def sum_cells(self, left, right):
        """Per cell the sum of `left` over its faces as left cell and of `right` as right cell."""
        out = torch.zeros((self.nc,) + left.shape[1:], dtype=F64, device=DEV)
        out.index_add_(0, self.L, left)
        out.index_add_(0, self.R[self.inner], right[self.inner])
        return out

    def neighbour(self, c, slot):
        """The cell across slot `slot` of cell c, or -1 (also for c = -1)."""
        e = self.face[c.clamp(min=0), slot]
        n = torch.where(self.L[e] == c, self.R[e], self.L[e])
        return torch.where((c >= 0) & (e >= 0), n, -1)

    def per_cell(self):
        """The reference layout's arrays of a quadrilateral mesh: neighbours (-1 at boundaries),
        outward normals, lengths and centre distances, 4 slots per cell."""
        e = self.face
        me = torch.arange(self.nc, device=DEV)[:, None]
        sign = torch.where(self.L[e] == me, 1.0, -1.0).to(F64)
        nbr = torch.where(self.L[e] == me, self.R[e], self.L[e])
        nrm = torch.stack([sign * self.nx[e], sign * self.ny[e]], 2).reshape(self.nc, 8)
        return dict(nbr=nbr, nrm=nrm, len=self.dl[e], dist=self.d.norm(dim=1)[e])


def _prims(U):
    """(rho, u, v, p, a) of conserved rows."""
    rho, u, v = U[:, 0], U[:, 1] / U[:, 0], U[:, 2] / U[:, 0]
    u = torch.where(u.abs() <= 1e-10, torch.zeros_like(u), u)
    v = torch.where(v.abs() <= 1e-10, torch.zeros_like(v), v)
    p = GM1 * (U[:, 3] - 0.5 * rho * (u * u + v * v))
    return torch.stack([rho, u, v, p, torch.sqrt(1.4 * p / rho)])


def _with_sound(W):
    return torch.cat([W[:4], torch.sqrt(1.4 * W[3:4] / W[0:1])])


def _energy(W):
    return W[3] / GM1 + 0.5 * W[0] * (W[1] ** 2 + W[2] ** 2)


def _slope(lim, a, b):
    z, pos = torch.zeros_like(a), a * b > 0
    if lim == "vanalbada":
        e = 1e-4
        return (a * (b * b + e) + b * (a * a + e)) / (a * a + b * b + 2 * e)
    if lim == "minmod":
        return torch.where(pos, torch.sign(b) * torch.minimum(a.abs(), b.abs()), z)
    return torch.where(pos, 2 * a * b / torch.where(pos, a + b, torch.ones_like(a)), z)


def _weno(s, shift):
    """WENO-JS edge value of the stencil s[0..4] centred on s[2]."""
    a, b, c, d, e = s
    b2 = 13 / 12 * (a - 2 * b + c) ** 2 + 0.25 * (a - 4 * b + 3 * c) ** 2
    b1 = 13 / 12 * (b - 2 * c + d) ** 2 + 0.25 * (b - d) ** 2
    b0 = 13 / 12 * (c - 2 * d + e) ** 2 + 0.25 * (3 * c - 4 * d + e) ** 2
    if shift == 0:
        w, v = (0.3, 0.6, 0.1), ((2 * c + 5 * d - e) / 6, (-b + 5 * c + 2 * d) / 6, (2 * a - 7 * b + 11 * c) / 6)
    else:
        w, v = (0.1, 0.6, 0.3), ((11 * c - 7 * d + 2 * e) / 6, (2 * b + 5 * c - d) / 6, (-a + 5 * b + 2 * c) / 6)
    al = [x / (1e-6 + y) ** 2 for x, y in zip(w, (b0, b1, b2))]
    t = al[0] + al[1] + al[2]
    return torch.where(t < 1e-6, (v[0] + v[1] + v[2]) / 3, (al[0] * v[0] + al[1] * v[1] + al[2] * v[2]) / t)


class _Exact:
    """The scheme of a configuration on one mesh, in plain torch."""

    def __init__(self, pts, cells, kw):
        self.g, self.kw = _Faces(pts, cells), kw
        g, self.psi = self.g, None
        d2 = (g.d ** 2).sum(1)
        M = g.sum_cells(*[torch.stack([g.d[:, 0] ** 2, g.d[:, 0] * g.d[:, 1], g.d[:, 1] ** 2], 1) / d2[:, None]] * 2)
        det = M[:, 0] * M[:, 2] - M[:, 1] ** 2
        inv = torch.stack([M[:, 2], -M[:, 1], M[:, 0]], 1) / det[:, None]
        vec = lambda c: torch.stack([inv[c, 0] * g.d[:, 0] + inv[c, 1] * g.d[:, 1],  # noqa: E731
                                     inv[c, 1] * g.d[:, 0] + inv[c, 2] * g.d[:, 1]], 1) / d2[:, None]
        self.wL, self.wR = vec(g.L), vec(g.R.clamp(min=0))
        if kw["order"] == 3:
            back = lambda c, s: torch.where(g.nf[c.clamp(min=0)] == 4, g.neighbour(c, (s + 2) % 4), -1)  # noqa: E731

            def beyond(c, s):
                one = back(c, s)
                slot = (g.face[one.clamp(min=0)] == g.face[c, (s + 2) % 4][:, None]).int().argmax(1)
                return one, back(one, slot)

            l1, l2 = beyond(g.L, g.sL)
            r1, r2 = beyond(g.R.clamp(min=0), g.sR)
            self.line = torch.stack([l2, l1, r1, r2])
            self.on_line = g.inner & (self.line >= 0).all(0)

    def ghost(self, W):
        """Ghost primitives of face states W (only the boundary faces' entries are used)."""
        g, out = self.g, W.clone()
        fs = self.kw["fs"]
        for kind, bc in enumerate(self.kw["bc"], 1):
            m = (g.kind == kind) & ~g.inner
            rho, u, v, p = (W[q][m] for q in range(4))
            if bc == "freestream":
                new = [torch.full_like(rho, float(q)) for q in fs]
            elif bc == "inlet_ref":
                new = [torch.full_like(rho, float(fs[0])), u, v, torch.full_like(rho, float(fs[3]))]
            elif bc == "noslip_wall":
                new = [rho, -u, -v, p]
            elif bc in ("wall", "symmetry"):
                vn = 2 * (u * g.nx[m] + v * g.ny[m])
                new = [rho, u - vn * g.nx[m], v - vn * g.ny[m], p]
            else:
                continue
            for q in range(4):
                out[q][m] = new[q]
        return _with_sound(out)

    def gradients(self, W, ghosts):
        g = self.g
        WL = W[:4, g.L].T
        WR = torch.where(g.inner, W[:4, g.R.clamp(min=0)], ghosts[:4]).T
        if self.kw["gradient"] == "wlsq":
            dW = (WR - WL)[:, :, None]
            return g.sum_cells(dW * self.wL[:, None], dW * self.wR[:, None])
        f = 0.5 * (WL + torch.where(g.inner[:, None], WR, WL))
        n = torch.stack([g.nx * g.dl, g.ny * g.dl], 1)
        f = f[:, :, None] * n[:, None]
        return g.sum_cells(f, -f) / g.area[:, None, None]

    def flux(self, L, R):
        """Face flux per unit length of primitive states (rho, u, v, p, a)."""
        g, kind = self.g, self.kw["flux"]
        nx, ny = g.nx, g.ny
        side = lambda W: (W[1] * nx + W[2] * ny, _energy(W))  # noqa: E731
        (qL, EL), (qR, ER) = side(L), side(R)
        cons = lambda W, E: torch.stack([W[0], W[0] * W[1], W[0] * W[2], E])  # noqa: E731
        phys = lambda W, q, E: torch.stack([W[0] * q, W[0] * W[1] * q + W[3] * nx, W[0] * W[2] * q + W[3] * ny,  # noqa: E731
                                            (E + W[3]) * q])
        UL, UR, FL, FR = cons(L, EL), cons(R, ER), phys(L, qL, EL), phys(R, qR, ER)
        sl, sr = torch.sqrt(L[0]), torch.sqrt(R[0])
        avg = lambda x, y: (x * sl + y * sr) / (sl + sr)  # noqa: E731
        if kind == "llf":
            s = torch.maximum(qL.abs() + L[4], qR.abs() + R[4])
            return 0.5 * (FL + FR) - 0.5 * s * (UR - UL)
        if kind == "hllc":
            u, a = avg(qL, qR), avg(L[4], R[4])
            SL, SR = torch.minimum(qL - L[4], u - a), torch.maximum(qR + R[4], u + a)
            den = L[0] * (SL - qL) - R[0] * (SR - qR)
            S = (R[3] - L[3] + L[0] * qL * (SL - qL) - R[0] * qR * (SR - qR)) / den

            def star(W, U, F, q, E, SK):
                f = W[0] * (SK - q) / (SK - S)
                Us = torch.stack([f, f * (W[1] + (S - q) * nx), f * (W[2] + (S - q) * ny),
                                  f * (E / W[0] + (S - q) * (S + W[3] / (W[0] * (SK - q))))])
                return F + SK * (Us - U)

            mid = torch.where(S >= 0, star(L, UL, FL, qL, EL, SL), star(R, UR, FR, qR, ER, SR))
            return torch.where(SL >= 0, FL, torch.where(SR <= 0, FR, mid))
        HL, HR = (EL + L[3]) / L[0], (ER + R[3]) / R[0]
        u, v, H = avg(L[1], R[1]), avg(L[2], R[2]), avg(HL, HR)
        ke = 0.5 * (u * u + v * v)
        a = torch.sqrt(GM1 * (H - ke))
        if kind == "ausm":
            ML, MR = qL / a, qR / a
            sup = lambda M: M.abs() >= 1  # noqa: E731
            Mp = torch.where(sup(ML), ML.clamp(min=0), 0.25 * (ML + 1) ** 2)
            Mm = torch.where(sup(MR), MR.clamp(max=0), -0.25 * (MR - 1) ** 2)
            Pp = torch.where(sup(ML), (ML > 0).to(F64), 0.25 * (ML + 1) ** 2 * (2 - ML))
            Pm = torch.where(sup(MR), (MR < 0).to(F64), 0.25 * (MR - 1) ** 2 * (2 + MR))
            M, p = Mp + Mm, Pp * L[3] + Pm * R[3]
            up = M >= 0
            w = lambda x, y: torch.where(up, x, y)  # noqa: E731
            mf = M * a * w(L[0], R[0])
            return torch.stack([mf, mf * w(L[1], R[1]) + p * nx, mf * w(L[2], R[2]) + p * ny, mf * w(HL, HR)])
        q, t, r = nx * u + ny * v, -ny * u + nx * v, torch.sqrt(L[0] * R[0])
        dr, du, dv, dp = R[0] - L[0], R[1] - L[1], R[2] - L[2], R[3] - L[3]
        dq, dt = nx * du + ny * dv, -ny * du + nx * dv
        s1, s4 = (dp - r * a * dq) / (2 * a * a), (dp + r * a * dq) / (2 * a * a)
        fix = lambda x: torch.where(x < 0.1 * a, 0.5 * (x * x / (0.1 * a) + 0.1 * a), x)  # noqa: E731
        t1, t2, t3, t4 = fix((q - a).abs()) * s1, q.abs() * (dr - dp / (a * a)), q.abs() * r * dt, fix((q + a).abs()) * s4
        D = torch.stack([t1 + t2 + t4, t1 * (u - nx * a) + t2 * u - t3 * ny + t4 * (u + nx * a),
                         t1 * (v - ny * a) + t2 * v + t3 * nx + t4 * (v + ny * a),
                         t1 * (H - a * q) + t2 * ke + t3 * t + t4 * (H + a * q)])
        if not self.kw["roe_bdiss"]:
            D = D * g.inner
        return 0.5 * (FL + FR) - 0.5 * D

    def viscous_flux(self, WL, WR, GL, GR):
        g, kw = self.g, self.kw
        GR = torch.where(g.inner[:, None, None], GR, GL)
        T = lambda W: W[3] / (W[0] * kw["r_gas"])  # noqa: E731
        gT = lambda W, G: (G[:, 3] - (W[3] / W[0])[:, None] * G[:, 0]) / (W[0] * kw["r_gas"])[:, None]  # noqa: E731
        dist = g.d.norm(dim=1)
        t = g.d / dist[:, None]

        def at_face(a, b, pl, pr):
            m = 0.5 * (a + b)
            return m + ((pr - pl) / dist - (m * t).sum(1))[:, None] * t

        du, dv = at_face(GL[:, 1], GR[:, 1], WL[1], WR[1]), at_face(GL[:, 2], GR[:, 2], WL[2], WR[2])
        dT = at_face(gT(WL, GL), gT(WR, GR), T(WL), T(WR))
        mu = kw["mu"]
        k = mu * 1.4 * kw["r_gas"] / (GM1 * kw["prandtl"])
        txx, tyy = 2 / 3 * mu * (2 * du[:, 0] - dv[:, 1]), 2 / 3 * mu * (2 * dv[:, 1] - du[:, 0])
        txy = mu * (du[:, 1] + dv[:, 0])
        u, v = 0.5 * (WL[1] + WR[1]), 0.5 * (WL[2] + WR[2])
        return torch.stack([0 * u, txx * g.nx + txy * g.ny, txy * g.nx + tyy * g.ny,
                            (txx * u + txy * v + k * dT[:, 0]) * g.nx + (txy * u + tyy * v + k * dT[:, 1]) * g.ny])

    def residual(self, U, Uexit=None, first=None, freeze=0):
        """Net flux per cell, and the gradients; `first`: cells whose faces take first-order states."""
        g, kw = self.g, self.kw
        W = _prims(U)
        WL = W[:, g.L]
        gh = self.ghost(WL)
        exits = torch.zeros_like(g.inner)
        if Uexit is not None:
            for kind, bc in enumerate(kw["bc"], 1):
                exits |= ~g.inner & (g.kind == kind) & (bc == "exit")
            gh = torch.where(exits, _prims(Uexit)[:, g.L], gh)
        WR = torch.where(g.inner, W[:, g.R.clamp(min=0)], gh)
        fL, fR, G = WL, WR, None
        if kw["order"] >= 2:
            G = self.gradients(W, gh)
            GL, GR = G[g.L], G[g.R.clamp(min=0)]
            dp = WR[:4] - WL[:4]
            cc = [(x * g.d[:, None]).sum(2).T for x in (GL, GR)]
            sl = [_slope(kw["limiter"], 2 * c - dp, dp) for c in cc]
            if freeze == 2:
                sl = [p * c for p, c in zip(self.psi, cc)]
            elif freeze == 1:
                self.psi = [torch.where(c != 0, s / c, 0 * c).float().to(F64) for s, c in zip(sl, cc)]

            def side(c, w):
                ok = (w[0] > 0) & (w[3] > 0)
                return torch.where(ok, _with_sound(torch.where(ok, w, c[:4])), c)

            fL = side(WL, WL[:4] + 0.5 * sl[0])
            fR = torch.where(g.inner, side(WR, WR[:4] - 0.5 * sl[1]), self.ghost(fL))
        if kw["order"] == 3:
            s = [U[c.clamp(min=0)].T for c in (self.line[0], self.line[1], g.L, g.R, self.line[2], self.line[3])]
            for shift, lo, c in ((0, 0, WL), (1, 1, WR)):
                w = _prims(_weno(s[lo:lo + 5], shift).T)
                w = torch.where((w[0] > 0) & (w[3] > 0), w, c)
                if shift == 0:
                    fL = torch.where(self.on_line, w, fL)
                else:
                    fR = torch.where(self.on_line, w, fR)
        if first is not None:
            m = first[g.L] | (g.inner & first[g.R.clamp(min=0)])
            fL, fR = torch.where(m, WL, fL), torch.where(m, WR, fR)
        F = self.flux(fL, fR)
        if kw.get("viscous", "off") != "off":
            F = F - self.viscous_flux(WL, WR, GL, GR)
        F = (F * g.dl).T
        return g.sum_cells(F, -F), G

    def time_step(self, U):
        g, kw, W = self.g, self.kw, _prims(U)
        rad = lambda c: ((W[1][c] * g.nx + W[2][c] * g.ny).abs() + W[4][c]) * g.dl  # noqa: E731
        den = g.sum_cells(rad(g.L), rad(g.R.clamp(min=0)))
        if kw.get("viscous", "off") != "off":
            s = g.sum_cells(g.dl ** 2, g.dl ** 2)
            den = den + 4 * torch.clamp(4 / (3 * W[0]), min=1.4 / W[0]).maximum(1.4 / W[0]) * kw["mu"] / kw["prandtl"] * s / g.area
        return kw["cfl"] * g.area / den

    def inadmissible(self, Us, Uo):
        """Cells the positivity fallback recomputes: stage input Us, stage output Uo."""
        g, bad = self.g, None
        for q in (0, 3):
            w = _prims(Us)[q].float().to(F64)
            l, r = g.L[g.inner], g.R[g.inner]
            lo, hi = w.clone(), w.clone()
            for x, y in ((l, r), (r, l)):
                lo = lo.scatter_reduce(0, x, w[y], "amin")
                hi = hi.scatter_reduce(0, x, w[y], "amax")
            o = _prims(Uo)[q]
            m = torch.maximum(1e-3 * hi.abs(), 1e-3 * (hi - lo))
            out = ~(o > 0)
            if self.kw["positivity"] == 1:
                out |= ~((o >= lo - m) & (o <= hi + m))
            bad = out if bad is None else bad | out
        return bad

    def step(self, U, freeze=0):
        """One native step; returns the new state and Error[0..3]."""
        kw, A = self.kw, self.g.area
        dt = self.time_step(U)
        h = ((dt if kw["lts"] else dt.min()) / A)[:, None]
        us, acc = U, 0
        for k in range(4 if kw["rk"] == 4 else 3):
            def out(r):
                if kw["rk"] == 4:
                    return (U - 0.5 * h * r, U - 0.5 * h * r, U - h * r, U - h / 6 * (acc + r))[k]
                e = us - h * r
                return (U - h * r, 0.75 * U + 0.25 * e, U / 3 + 2 / 3 * e)[k]

            r, _ = self.residual(us, freeze=freeze)
            new = out(r)
            if kw.get("positivity"):
                bad = self.inadmissible(us, new)
                if bool(bad.any()):
                    r, _ = self.residual(us, first=bad, freeze=freeze)
                    new = out(r)
            acc = r if k == 0 else acc + 2 * r
            us = new
        return us, _error(us - U, U)

    def reference_step(self, U):
        """One iteration of the reference: delta-form TVD-RK3, each stage's own global time step."""
        ia, us = (1.0 / self.g.area)[:, None], U
        for k in range(3):
            r, _ = self.residual(us, Uexit=U)
            d = self.time_step(us).min() * ia * r
            us = (U - d, 0.25 * (us + 3 * U - d), U + 2 / 3 * (us - U - d))[k]
        return us


def _error(d, u):
    t = torch.where(d < 1e-9, d.abs(), d.abs() / u)
    return torch.sqrt((t * t).sum(0))


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        return globals()["_exact_" + kind](case, seed)


def _exact_march(case, seed):
    pts, cells = _points_cells(case["mesh"], case["n"], _quads(case))
    if len(cells) * case["nsteps"] > 3000000:
        return None  # takes too long
    # the outputs' row order: the handle's renumbering (host arrays only)
    perm = torch.as_tensor(_mesh(case["mesh"], case["n"], _quads(case), case["shape"], False).permutation(), device=DEV).long()
    e, U, err = _Exact(pts, cells, _flow_setup(case)), _state(case, seed), None
    for _ in range(case["nsteps"]):
        if case["ref_mode"]:
            U = e.reference_step(U)
        else:
            U, err = e.step(U)
    out = dict(U=U[perm])
    if case["call"] == "steady":
        out.update(steps=None, error=err)
    return out


def _exact_residual(case, seed):
    pts, cells = _points_cells(case["mesh"], case["n"], _quads(case))
    e, U = _Exact(pts, cells, _flow_setup(case)), _state(case, seed)
    R, G = e.residual(U)
    out = dict(R=R, dt=e.time_step(U))
    if G is not None:
        out["grad"] = G.reshape(-1, 8)
    return out


def _exact_batch(case, seed):
    cs = _ramps(case["instances"], case["min_cells"], case["max_cells"])
    if sum(len(c.mesh.cells) for c in cs) * case["nsteps"] > 20000000:
        return None  # takes too long
    out, err = [], []
    for i, (c, U) in enumerate(zip(cs, _batch_states(case, seed))):
        e = _Exact(c.mesh.points, c.mesh.cells, dict(_batch_scheme(), fs=tuple(float(v) for v in c.fs)))
        for k in range(case["nsteps"]):
            U, er = e.step(U, freeze=0 if i % 2 == 0 else 1 if k == 0 else 2)
        out.append(U)
        err.append(er[0])
    return dict(U=out, error0=torch.stack(err), steps=None, status=None)


def _exact_wrappers(case, seed):
    s = _prepare_wrappers(case, seed)
    pts, cells = _points_cells("bump", case["n"], True)
    g = _Faces(pts, cells)
    U, nb, dist, N = s["U"], s["nb"].long(), s["dist"], s["N"]
    there = (nb >= 0)[..., None]
    dU = U[nb.clamp(min=0)] - U[:, None]
    fwd = 0.5 * dU / dist[..., None]
    opp = torch.where(there.roll(2, 1), -fwd.roll(2, 1), torch.zeros_like(fwd))
    r = opp / fwd
    phi = torch.where(there & (fwd.abs() >= 1e-12) & (r > 0), 2 * r / (1 + r), torch.zeros_like(fwd))
    back = (nb[nb.clamp(min=0)] == torch.arange(N, device=DEV)[:, None, None]).int().argmax(2)
    pR = phi[nb.clamp(min=0), back]
    QL = U[:, None] + torch.where(there, 0.25 * phi * dU, 0 * phi)
    QR = torch.where(there, U[nb.clamp(min=0)] - 0.25 * pR * dU, U[:, None])
    F = torch.zeros(N, 4, 4, dtype=F64, device=DEV)
    W = _prims(U)
    for k in range(4):
        e = _Exact.__new__(_Exact)
        e.g, e.kw = _Slot(g.nx, nb[:, k], s["nrm"][:, 2 * k], s["nrm"][:, 2 * k + 1]), dict(flux=case["flux"], roe_bdiss=1)
        f = e.flux(W, W[:, nb[:, k].clamp(min=0)])
        F[:, k] = torch.where(there[:, k], (f * s["len"][:, k]).T, F[:, k])
    return dict(phi=phi, QL=QL, QR=QR, F=F, Urk=U - 1e-5 * s["ia"][:, None] * s["net"])


class _Slot:
    """One face slot of every cell, as `_Exact.flux` reads a face list."""

    def __init__(self, like, nbr, nx, ny):
        self.nx, self.ny, self.inner = nx, ny, nbr >= 0


def _layers(m):
    W, b = (torch.as_tensor(v, device=DEV, dtype=F64) for v in m.get_params())
    dims = [(4 if k == 0 else m.width, 4 if k == m.depth else m.width) for k in range(m.depth + 1)]
    Ws, bs, iw, ib = [], [], 0, 0
    for k, n in dims:
        Ws.append(W[iw:iw + k * n].reshape(n, k).clone())
        bs.append(b[ib:ib + n].clone())
        iw, ib = iw + k * n, ib + n
    return Ws, bs


def _forward(Ws, bs, X):
    xs, zs = [X], []
    for k, (w, b) in enumerate(zip(Ws, bs)):
        zs.append(xs[-1] @ w.T + b)
        if k < len(Ws) - 1:
            xs.append(torch.nn.functional.silu(zs[-1]))
    return xs, zs


def _norm(m):
    return [torch.as_tensor(v, device=DEV, dtype=F64) for v in m.norm]


def _exact_mlp_predict(case, seed):
    m = _network(case, seed, 512)
    im, sc, om, os_ = _norm(m)
    X = torch.as_tensor(_samples(case["rows"], seed)[0], device=DEV, dtype=F64)
    Ws, bs = _layers(m)
    return torch.cat([_forward(Ws, bs, (x - im) * sc)[1][-1] / os_ + om for x in X.split(1 << 17)])


def _exact_mlp_train(case, seed):
    m = _network(case, seed, 512)
    im, sc, om, os_ = _norm(m)
    feat, targ = (torch.as_tensor(v, device=DEV, dtype=F64) for v in _samples(case["samples"], seed))
    X, T = (feat - im) * sc, (targ - om) * os_
    Ws, bs = _layers(m)
    par = Ws + bs
    m1, m2 = [torch.zeros_like(p) for p in par], [torch.zeros_like(p) for p in par]
    B, n, hist = case["batch"], case["nsteps"], None
    mask = (1 << 64) - 1
    for s in range(n):
        # the minibatch: SplitMix64 of (seed, step, row), as MLP.train documents it
        with np.errstate(over="ignore"):
            z = np.uint64(1) + np.uint64(0x9E3779B97F4A7C15) * (np.uint64(s * B & mask) + np.arange(1, B + 1, dtype=np.uint64))
            z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
            z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
            z ^= z >> np.uint64(31)
        idx = torch.as_tensor((z % np.uint64(len(X))).astype(np.int64), device=DEV)
        xs, zs = _forward(Ws, bs, X[idx])
        E = zs[-1] - T[idx]
        if hist is None:
            hist = (E * E).mean()
        dZ, gW, gb = 2 * E / E.numel(), [None] * len(Ws), [None] * len(Ws)
        for k in range(len(Ws) - 1, -1, -1):
            gW[k], gb[k] = dZ.T @ xs[k], dZ.sum(0)
            if k:
                sg = torch.sigmoid(zs[k - 1])
                dZ = (dZ @ Ws[k]) * (sg * (1 + zs[k - 1] * (1 - sg)))
        lr = 5e-5 + (2e-3 - 5e-5) * (0.5 * (1 + math.cos(math.pi * s / (n - 1))) if n > 1 else 1.0)
        for p, a, b, gr in zip(par, m1, m2, gW + gb):
            a.mul_(0.9).add_(gr, alpha=0.1)
            b.mul_(0.999).add_(gr * gr, alpha=0.001)
            p -= lr * (a / (1 - 0.9 ** (s + 1))) / (torch.sqrt(b / (1 - 0.999 ** (s + 1))) + 1e-8)
    return dict(W=torch.cat([w.reshape(-1) for w in Ws]), b=torch.cat(bs), loss=hist.reshape(1))
