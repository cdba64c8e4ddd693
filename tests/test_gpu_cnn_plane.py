"""The convolutions by runs of 256 voxels and the weight gradient by padded
x-rows at grids that are no multiple of 16 (and the smallest), against the
voxel-tile kernels that serve any grid."""
import numpy as np
import pytest

from distributednavierstokes_amd.cnn import SFSNet
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
