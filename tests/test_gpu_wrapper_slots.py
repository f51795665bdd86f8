"""The reference-layout wrappers, one thread per face slot, at the edges of their launches (cell
counts around a block, blocks that are no multiple of a cell's four slots) and on arrays aligned to
one value only, against the oracle's restatement, bit for bit."""
import ctypes

import numpy as np
import pytest

from cfd_solver_withcuda_amd._lib import DeviceArray, lib
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

_dp = ctypes.POINTER(ctypes.c_double)
_ip = ctypes.POINTER(ctypes.c_int)


class Shifted:
    """A device copy of `a` that starts `off` values into its allocation."""

    def __init__(self, a, off):
        self.a = np.ascontiguousarray(a)
        self.off = off
        self.dev = DeviceArray(np.concatenate([np.zeros(off, a.dtype), self.a.ravel(), np.zeros(4, a.dtype)]))

    @property
    def ptr(self):
        return ctypes.c_void_p(self.dev.ptr.value + self.off * self.a.itemsize)

    def get(self):
        return self.dev.get()[self.off: self.off + self.a.size].reshape(self.a.shape)


def d(a):
    return a.ctypes.data_as(_dp)


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("N,block", [(1, 64), (63, 256), (65, 100), (257, 33), (1000, 1024)])
def test_slots_vs_oracle(N, block, off):
    print(f"case N={N} block={block} off={off}", flush=True)
    L, orc = lib(), Oracle().lib
    r = np.random.default_rng(N)
    # a ring of cells: slot 0/2 the next/previous cell, slot 1/3 outside
    nb = np.full((N, 4), -1, np.int32)
    if N > 1:
        nb[:, 0], nb[:, 2] = (np.arange(N) + 1) % N, (np.arange(N) - 1) % N
    rho, u, v, p = (r.uniform(0.5, 1.5, N) for _ in range(4))
    U = np.stack([rho, rho * u, rho * v, p / (1.4 - 1.0) + 0.5 * rho * (u * u + v * v)], 1)
    P = np.stack([rho, u, v, p, p / (287.0 * rho), np.sqrt(1.4 * p / rho)], 1)
    th = r.uniform(0, 6, (N, 4))
    nrm = np.stack([np.cos(th), np.sin(th)], 2).reshape(N, 8)
    ln, dist, phi = r.uniform(0.5, 1.5, (N, 4)), r.uniform(0.5, 1.5, (N, 4)), r.uniform(0, 1, (N, 4, 4))
    g = {k: Shifted(np.ascontiguousarray(x), off)
         for k, x in dict(U=U, P=P, nb=nb, nrm=nrm, ln=ln, dist=dist, phi=phi, o1=np.full((N, 4, 4), 7.0),
                          o2=np.full((N, 4, 4), 7.0)).items()}
    c = ctypes.c_double

    def same(*pairs):
        for got, ref in pairs:
            assert np.array_equal(got.get(), ref)

    for scheme, name in enumerate(("launch_roe_flux", "launch_hllc_flux", "launch_llf_flux")):
        g["o1"] = Shifted(np.full((N, 4, 4), 7.0), off)
        assert getattr(L, name)(g["U"].ptr, g["P"].ptr, g["nb"].ptr, g["nrm"].ptr, g["ln"].ptr, g["o1"].ptr, N, c(1.4),
                                block, None) == 0
        ref = np.full((N, 4, 4), 7.0)
        orc.rl_flux(scheme, d(U), d(P), nb.ctypes.data_as(_ip), d(nrm), d(ln), d(ref), N, 1.4)
        same((g["o1"], ref))
    assert L.launch_vanleer_limiter(g["U"].ptr, g["nb"].ptr, g["dist"].ptr, g["o1"].ptr, N, c(0.5), block, None) == 0
    ref = np.zeros((N, 4, 4))
    orc.rl_limiter(d(U), nb.ctypes.data_as(_ip), d(dist), d(ref), N, 0.5, 1, 0)
    same((g["o1"], ref))
    assert L.launch_muscl_reconstruction(g["U"].ptr, g["nb"].ptr, g["dist"].ptr, g["phi"].ptr, g["o1"].ptr, g["o2"].ptr,
                                         N, c(0.5), block, None) == 0
    QL, QR = np.zeros((N, 4, 4)), np.zeros((N, 4, 4))
    orc.rl_muscl(d(U), nb.ctypes.data_as(_ip), d(dist), d(phi), d(QL), d(QR), N, 0.5)
    same((g["o1"], QL), (g["o2"], QR))
    assert L.launch_barth_jespersen_limiter(g["U"].ptr, g["nb"].ptr, g["dist"].ptr, g["phi"].ptr, g["o1"].ptr, N, block,
                                            None) == 0
    ref = np.zeros((N, 4, 4))
    orc.rl_bj(d(U), nb.ctypes.data_as(_ip), d(dist), d(phi), d(ref), N)
    same((g["o1"], ref))
