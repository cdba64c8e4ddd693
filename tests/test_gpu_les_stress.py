"""The stress that the LES adds to the products (output convolution with dx as
columns, planar and scaled) against the voxel-tile convolutions and the pass
that reorders their result."""
import numpy as np
import pytest

import distributednavierstokes_amd as dns
from distributednavierstokes_amd import _lib
from distributednavierstokes_amd._lib import check, dptr
from distributednavierstokes_amd.cnn import SFSNet
from distributednavierstokes_amd.spectral import DeviceState

pytestmark = pytest.mark.gpu


# compile-time widths (16, 32, 64); rows that fill a block (64), part of one (24, 36, 50), one row per block (144)
@pytest.mark.parametrize("n", [16, 24, 32, 36, 50, 64, 144])
@pytest.mark.parametrize("T", [np.float32, np.float64])
def test_stress_against_voxel_tiles(n, T, monkeypatch):
    """A step of Δt = 0 keeps the velocity, whatever the stress, so both forms
    see the same network inputs and (the convolutions accumulate in one order)
    the same hidden activations: what differs is the order of the FP32 sums of
    the last layer, 1e-6 of the norm as in the other comparisons of its sums.
    FP32 handles round the stress and its transform once more: 2e-6."""
    tau = []
    for kind in (None, "direct"):
        if kind:
            monkeypatch.setenv("DNS_CNN_CONV", kind)
        s = dns.spectral_setup(n=n, visc=1e-2, T=T)
        dns.spectral_randomfield_(DeviceState(s), s, totalenergy=1.0, kpeak=2, seed=3)
        net = SFSNet(M=n, batch=1, seed=0)
        net.set_params((np.random.default_rng(n).standard_normal(net.nparams) * 0.08).astype(np.float32))
        net.scales = (0.7, 0.013)
        check(_lib.lib().dns_les_closure_step(s.handle, net.handle, 0.0, None))
        t = np.zeros(s.state_shape[:3] + (6,), dtype=np.complex128, order="F")
        check(_lib.lib().dns_sfs_get(s.handle, None, dptr(t)))
        tau.append(t)
    for c in range(6):
        err = np.linalg.norm(tau[0][..., c] - tau[1][..., c]) / np.linalg.norm(tau[1][..., c])
        print(f"LES stress n={n} {T.__name__} component {c}: {err:.2e}", flush=True)
        assert err <= (1e-6 if T == np.float64 else 2e-6)
