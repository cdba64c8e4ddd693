"""One set of network values: what forward, evaluate and predict return is
what the training loss is made of, and what the voxel-tile convolutions give."""
import numpy as np
import pytest

from distributednavierstokes_amd.cnn import SFSNet

pytestmark = pytest.mark.gpu


def network(M, B=1):
    net = SFSNet(M=M, batch=B, seed=0)
    net.set_params((np.random.default_rng(M).standard_normal(net.nparams) * 0.08).astype(np.float32))
    return net


def pair(M, seed=1):
    rng = np.random.default_rng(seed)
    return rng.standard_normal((M, M, M, 3)).astype(np.float32), (rng.standard_normal((M, M, M, 6)) * 0.1).astype(np.float32)


@pytest.mark.parametrize("M", [4, 16, 20, 32, 36, 64])
def test_evaluation_is_the_training_loss(M):
    """The same sample, the same kernels in the same order: equal to the last bit."""
    net = network(M)
    u, t = pair(M)
    net.add_sample(u, t)
    net.fit_scales()
    before = net.evaluate(0, 1)
    p = net.predict(0)
    assert net.train(1, lr=0.0)[0] == before
    su, st = net.scales
    y = net.forward((u / np.float32(su)).transpose(2, 1, 0, 3)[None])[0].transpose(2, 1, 0, 3)
    # su divides here and its FP32 inverse multiplies there: inputs may round to another BF16 value
    assert np.linalg.norm(y * st - p) <= 3e-2 * np.linalg.norm(p)


@pytest.mark.parametrize("M", [2, 5, 16, 17, 20, 32, 36, 64])
def test_forward_is_the_voxel_tiles(M, monkeypatch):
    """Products accumulate in the same order in the convolutions by runs of
    256 voxels and by voxel tiles: the same values to the last bit."""
    x = np.random.default_rng(3).standard_normal((1, M, M, M, 3)).astype(np.float32)
    got = network(M).forward(x)
    monkeypatch.setenv("DNS_CNN_CONV", "direct")
    assert np.array_equal(got, network(M).forward(x))
