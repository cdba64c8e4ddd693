"""The SFS buffer of an LES handle after closure steps: ``dns_sfs_get``,
``dns_sfs_physical`` and ``dns_sfs_append`` hand out the learned stress of
the last stage, with or without an earlier sample, until a sample replaces it."""
import numpy as np
import pytest

import distributednavierstokes_amd as dns
from distributednavierstokes_amd import _lib
from distributednavierstokes_amd._lib import check, dptr
from distributednavierstokes_amd.cnn import SFSNet
from distributednavierstokes_amd.les import lessampler
from distributednavierstokes_amd.spectral import DeviceState

pytestmark = pytest.mark.gpu


def get(s):
    ub = np.zeros(s.state_shape, dtype=np.complex128, order="F")
    tau = np.zeros(s.state_shape[:3] + (6,), dtype=np.complex128, order="F")
    check(_lib.lib().dns_sfs_get(s.handle, dptr(ub), dptr(tau)))
    return ub, tau


def physical(s):
    n = s.n
    ub, tau = np.zeros((n, n, n, 3), order="F"), np.zeros((n, n, n, 6), order="F")
    check(_lib.lib().dns_sfs_physical(s.handle, dptr(ub), dptr(tau)))
    return ub, tau


def network(n, seed=4):
    net = SFSNet(M=n, batch=1, seed=0)
    net.set_params((np.random.default_rng(seed).standard_normal(net.nparams) * 0.08).astype(np.float32))
    net.scales = (0.7, 0.013)
    return net


def predicted(net, v):
    """The network's stress of a physical velocity through ``predict`` (FP32, physical units)."""
    other = network(net.M)
    other.add_sample(v, np.zeros(v.shape[:3] + (6,)))
    return other.predict(0).astype(np.float64)


# 18: block x pass (the step itself transforms the stress); the others add it in physical space
@pytest.mark.parametrize("n", [18, 32, 36, 50])
@pytest.mark.parametrize("T", [np.float32, np.float64])
def test_stress_after_step(n, T):
    """At Δt = 0 all stages see the same velocity up to rounding, so the stress
    is the network's at the state.  The network's BF16 inputs may round the
    other way where the projection of a stage moved a velocity by its own
    rounding: 3e-2 of the norm, the bound of the closure tests; against the
    physical stress the same buffer gives, the transforms' 1e-12 and 2e-5."""
    tol = 2e-5 if T == np.float32 else 1e-12
    s = dns.spectral_setup(n=n, visc=1e-2, T=T)
    dns.spectral_randomfield_(DeviceState(s), s, totalenergy=1.0, kpeak=2, seed=n)
    net = network(n)
    check(_lib.lib().dns_les_closure_step(s.handle, net.handle, 0.0, None))
    ub, tau = get(s)
    assert np.array_equal(ub, s.download())
    v, t = physical(s)
    ref = predicted(net, v)
    tools = dns.spectral_setup(n=n, visc=1e-2, T=T)
    full = np.zeros_like(tau)
    for c in (0, 3):
        w = np.zeros(s.state_shape, dtype=np.complex128, order="F")
        full[..., c:c + 3] = dns.phys_to_spec_(w, np.asfortranarray(ref[..., c:c + 3]), tools)
    err = np.linalg.norm(tau - full) / np.linalg.norm(full)
    print(f"n={n} {T.__name__}: stress after the step {err:.2e}", flush=True)
    assert err <= 3e-2
    # spectral and physical copies are one field
    back = np.zeros((n, n, n, 3), order="F")
    for c in (0, 3):
        dns.spec_to_phys_(back, np.asfortranarray(tau[..., c:c + 3]), tools)
        assert np.abs(back - t[..., c:c + 3]).max() <= tol * np.abs(t).max()
    # and the pair that a network's dataset gets
    other = network(n)
    check(_lib.lib().dns_sfs_append(s.handle, other.handle))
    assert other.nsamples == 1
    su, st = other.fit_scales()
    assert abs(st - np.sqrt(np.mean(t ** 2))) <= 1e-5 * st
    assert abs(su - np.sqrt(np.mean(v ** 2))) <= 1e-5 * su


def test_newest_of_sample_and_step():
    """A step's stress replaces a sample's and the other way round."""
    big = dns.spectral_setup(n=48, visc=1e-2)
    dns.spectral_randomfield_(DeviceState(big), big, totalenergy=1.0, kpeak=3, seed=2)
    ls = lessampler(big, M=24)
    _, t0 = ls.sample().spectral()
    net = network(24)
    check(_lib.lib().dns_les_closure_step(ls.les.handle, net.handle, 1e-3, None))
    _, t1 = ls.spectral()
    assert np.linalg.norm(t1 - t0) > 0.1 * np.linalg.norm(t0)
    _, t2 = ls.sample().spectral()
    assert np.array_equal(t2, t0)
