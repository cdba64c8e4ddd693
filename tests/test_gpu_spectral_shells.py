"""Shell factors as kernel arguments (up to 16) or through the device buffer,
and the velocity bound of every x pass against the one the step reports."""
import math

import numpy as np
import pytest

import distributednavierstokes_amd as dns
from distributednavierstokes_amd import _lib
from distributednavierstokes_amd.spectral import DeviceState, _rescale, _shells

pytestmark = pytest.mark.gpu


# one, the last count passed as arguments, the first that is not
@pytest.mark.parametrize("nsh", [1, 2, 15, 16, 17])
@pytest.mark.parametrize("T", [np.float64, np.float32])
def test_rescale_counts(nsh, T):
    """Energies scale by the squared factors and other shells stay: FP64 1e-12, FP32 1e-5."""
    s = dns.spectral_setup(n=64, visc=1e-3, T=T)
    dns.spectral_randomfield_(DeviceState(s), s, totalenergy=1.0, kpeak=4, seed=1)
    before = np.array(_shells(s, range(0, 21)))
    f = {2 + q: 0.5 + 0.1 * q for q in range(nsh)}
    _rescale(s, f)
    after = np.array(_shells(s, range(0, 21)))
    want = np.array([f.get(q, 1.0) ** 2 for q in range(21)]) * before
    assert np.allclose(after, want, rtol=1e-12 if T is np.float64 else 1e-5, atol=0)


# block kernel, two-step lines, one wavefront per 512-point line; one and two reduction levels
@pytest.mark.parametrize("n,T", [(10, np.float64), (96, np.float64), (128, np.float32), (256, np.float64), (512, np.float64)])
def test_velocity_bound(n, T):
    """vsummax and the bound of the first stage's velocity differ by FFT rounding only."""
    s = dns.spectral_setup(n=n, visc=1e-3, T=T)
    dns.spectral_randomfield_(DeviceState(s), s, totalenergy=1.0, kpeak=2, seed=2)
    a, b = np.zeros(1), np.zeros(1)
    _lib.check(_lib.lib().dns_spec_vsummax(s.handle, _lib.dptr(a)))
    _lib.check(_lib.lib().dns_spec_step(s.handle, 1e-6, _lib.dptr(b)))
    assert a[0] > 0
    assert math.isclose(a[0], b[0], rel_tol=1e-12 if T is np.float64 else 1e-5)
