"""Two-step pencil passes of the spectral path (k_p2_back, k_p2_fwd,
k_p2_stage) against the oracle's transforms, RHS, step and products."""
import numpy as np
import pytest

import distributednavierstokes_amd as dns
from distributednavierstokes_amd.problem import SpectralProblem
from oracle.oracle import OracleSpectral

pytestmark = pytest.mark.gpu


# the smallest length, lengths of the first radices 5 ... 16 (the larger ones run in
# test_gpu_spectral_shapes.py and the 512³ step), K below one tile, kcut far below n/3
@pytest.mark.parametrize("n,kcut", [(24, 8), (30, 10), (36, 3), (50, 16), (64, 21), (80, 26), (90, 30), (108, 36), (128, 20),
                                    (150, 50)])
@pytest.mark.parametrize("T", [np.float64, np.float32])
def test_p2_transforms_rhs_step_products(n, kcut, T):
    """Bounds as for the other transform tests: 1e-12 (FP64), 2e-5 (FP32)
    relative to the field's maximum."""
    tol = 1e-12 if T == np.float64 else 2e-5
    s = dns.spectral_setup(n=n, visc=5e-3, kcut=kcut, T=T)
    o = OracleSpectral(SpectralProblem(n=n, visc=5e-3, kcut=kcut))
    uh = o.randomfield(totalenergy=0.5, kpeak=2, seed=n)
    v = o.spec_to_phys(uh)
    vg = np.zeros_like(v, order="F")
    dns.spec_to_phys_(vg, uh, s)
    assert np.abs(vg - v).max() <= tol * np.abs(v).max()
    w = o.phys_to_spec(v)
    wg = np.zeros_like(uh)
    dns.phys_to_spec_(wg, v, s)
    assert np.abs(wg - w).max() <= tol * np.abs(w).max()
    du, _ = o.rhs(uh)
    dg = np.zeros_like(uh)
    dns.spectral_rhs_(dg, uh, s)
    assert np.abs(dg - du).max() <= tol * np.abs(du).max()
    ref, got = uh.copy(order="F"), uh.copy(order="F")
    o.step(ref, 1e-3)
    dns.spectral_step_(got, s, 1e-3)
    assert np.abs(got - ref).max() <= tol * np.abs(ref).max()
    if n <= 64:
        from distributednavierstokes_amd._lib import check, dptr, lib

        sig = o.products(uh)
        sg = np.zeros(uh.shape[:3] + (6,), dtype=np.complex128, order="F")
        s.upload(uh)
        check(lib().dns_spec_products(s.handle))
        check(lib().dns_spec_get_products(s.handle, dptr(sg)))
        assert np.abs(sg - sig).max() <= tol * np.abs(sig).max()


def test_slab_step_216():
    """A grid whose product pencils exceed the memory-side cache takes the z
    and x passes in 64-row slabs (here 64, 64 and 88 rows): step and max Σ|v|
    against the oracle."""
    n = 216
    s = dns.spectral_setup(n=n, visc=5e-3)
    o = OracleSpectral(SpectralProblem(n=n, visc=5e-3))
    ref = o.randomfield(totalenergy=0.5, kpeak=4, seed=1)
    got = ref.copy(order="F")
    vr = o.step(ref, 2e-3)
    vm = dns.spectral_step_(got, s, 2e-3)
    assert abs(vm - vr) <= 1e-12 * vr
    assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()
