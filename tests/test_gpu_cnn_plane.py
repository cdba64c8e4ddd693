"""The convolutions by runs of 256 voxels and the weight gradient by padded
x-rows at grids that are no multiple of 16 (and the smallest), against the
voxel-tile kernels that serve any grid."""
import numpy as np
import pytest

import distributednavierstokes_amd as dns
from distributednavierstokes_amd.cnn import SFSNet
from distributednavierstokes_amd.spectral import DeviceState
from oracle import oracle_cnn as oc

pytestmark = pytest.mark.gpu


def run(M, B):
    rng = np.random.default_rng(M)
    net = SFSNet(M=M, batch=B, seed=0)
    p = (rng.standard_normal(net.nparams) * 0.08).astype(np.float32)
    net.set_params(p)
    x = rng.standard_normal((B, M, M, M, 3)).astype(np.float32)
    t = (rng.standard_normal((B, M, M, M, 6)) * 0.1).astype(np.float32)
    return net.forward(x), net.loss_grad(x, t), net.grads()


# fewer voxels than a run, planes that end within one, rows around the 16-voxel
# slices of the gradient, the last M it takes and the first past it
@pytest.mark.parametrize("M,B", [(2, 3), (3, 2), (5, 2), (8, 2), (15, 2), (16, 1), (17, 2), (20, 1), (31, 1), (36, 2),
                                 (49, 1), (64, 1), (65, 1)])
def test_against_voxel_tiles(M, B, monkeypatch):
    """The convolutions sum in the same order: outputs to FP32 rounding of
    the last layer (1e-6).  The gradients' FP32 sums over up to 3·10⁵ voxels
    run in another order: 2e-5 of the norm per array."""
    y, loss, g = run(M, B)
    monkeypatch.setenv("DNS_CNN_CONV", "direct")
    monkeypatch.setenv("DNS_CNN_WGRAD", "row16")
    yr, lossr, gr = run(M, B)
    assert np.linalg.norm(y - yr) <= 1e-6 * np.linalg.norm(yr)
    assert abs(loss - lossr) <= 1e-6 * lossr
    off = 0
    for ci, co in oc.CH:
        for m in (27 * co * ci, co):
            assert np.linalg.norm(g[off:off + m] - gr[off:off + m]) <= 2e-5 * np.linalg.norm(gr[off:off + m])
            off += m


# planar FP32 and FP64 stress from the output convolution, whole rows of a block and not
@pytest.mark.parametrize("n", [16, 24, 30, 64])
@pytest.mark.parametrize("T", [np.float32, np.float64])
def test_les_increment_against_voxel_tiles(n, T, monkeypatch):
    """The change of an LES step with the stress written by the output
    convolution or by a pass over its result: to the bound of the network's
    BF16 inputs (3e-2, as against the FP64 restatement), since the velocity of
    the later stages passes through that rounding."""
    inc = []
    for kind in (None, "direct"):
        if kind:
            monkeypatch.setenv("DNS_CNN_CONV", kind)
        s = dns.spectral_setup(n=n, visc=1e-2, T=T)
        dns.spectral_randomfield_(DeviceState(s), s, totalenergy=1.0, kpeak=2, seed=3)
        net = SFSNet(M=n, batch=1, seed=0)
        net.set_params((np.random.default_rng(n).standard_normal(net.nparams) * 0.08).astype(np.float32))
        before = np.array(s.download())
        dns.spectral_solve_(uh=DeviceState(s), setup=s, tlims=(0.0, 1e-3), dt=1e-3, closure=net)
        inc.append(np.array(s.download()) - before)
    err = np.linalg.norm(inc[0] - inc[1]) / np.linalg.norm(inc[1])
    print(f"LES increment n={n} {T.__name__}: {err:.2e}", flush=True)
    assert err <= 3e-2
