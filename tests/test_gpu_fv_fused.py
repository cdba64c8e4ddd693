"""Explicit stages whose momentum kernel corrects the velocity as it reads it
(large grids), against the separate pressure-gradient passes behind the
slab-ordered momentum kernel."""
import math

import numpy as np
import pytest

import distributednavierstokes_amd as dns
from distributednavierstokes_amd.fv import ROCmBackend, Setup
from distributednavierstokes_amd.problem import FVProblem
from fvhelpers import channelproblem, randomfield, vzeros, zeros
from oracle.oracle import OracleFV

pytestmark = pytest.mark.gpu


# last x tile of 8 and of 44 columns, last y tile of 1 row, whole tiles; chunks
# cut short in z and a single one; walls and periodic y
@pytest.mark.parametrize("n,wall", [((200, 97, 90), True), ((300, 73, 80), True), ((128, 120, 108), False),
                                    ((192, 97, 90), True), ((512, 769, 4), True), ((128, 8, 1600), False)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_fused_stages(n, wall, precision, monkeypatch):
    """Two steps: 1e-12 of the largest value in FP64, 1e-5 with FP32 fields."""
    if wall:
        prob = channelproblem(n=n, visc=0.02, precision=precision, bodyforce=(1.0, 0.0, 0.0))
    else:
        prob = FVProblem(n=n, lims=((0.0, 2 * math.pi),) * 3, bc=("periodic",) * 3, visc=0.02, precision=precision)
    o = OracleFV(prob)
    u0 = randomfield(prob, seed=3, halo=o.exchange_halo_u)
    res = []
    for kind in (None, "slab"):
        if kind:
            monkeypatch.setenv("DNS_MOMENTUM", kind)
        s = Setup(prob, ROCmBackend())
        assert s.describe()["momentum"].startswith(kind or "lz")
        assert s.describe()["stages"].startswith("separate" if kind else "fused")
        s.upload_u([a.copy(order="F") for a in u0])
        dns._lib.check(dns._lib.lib().dns_fv_project(s.handle, dns._lib.FIELD["p"]))
        for nm in ("qx", "qy", "qz"):
            s.upload(nm, zeros(prob))
        dns.advance_cfl_(s, 0.3, 2)
        u = vzeros(prob)
        s.download_u(u)
        res.append((u, s.download("p")))
        del s
    (ua, pa), (ub, pb) = res
    tol = 1e-12 if precision == "fp64" else 1e-5
    for c in range(3):
        assert np.abs(ua[c] - ub[c]).max() <= tol * np.abs(ub[c]).max()
    if precision == "fp64":
        assert np.abs(pa - pb).max() <= 100 * tol * np.abs(pb).max()
