"""GPU tests of the weight gradient's tiles: every tile width (whole x-rows of 8 to 64 voxels, and two tiles a
row), channel counts that leave a 16-channel tile half empty or the last block of output channels short, odd
batches, against the FP64 oracle with the tolerances of its storage (activation gradients in bf16: 5e-2 in
relative L2 norm per layer, cosine above 0.998; one tap of 27 wrong would be 0.19)."""
import numpy as np
import pytest

from oracle import unet_oracle as U
from tests.test_gpu_net import _inputs

pytestmark = pytest.mark.gpu


def _net(g, levels, c0, B, seed):
    import homo3d_amd

    net = homo3d_amd.WarmStartNet(grid=g, levels=levels, base_channels=c0, batch=B, seed=3)
    theta = U.init_params(seed, levels, c0)
    theta += (0.02 * np.random.default_rng(seed + 1).standard_normal(theta.size)).astype(np.float32)
    net.set_params(theta)
    return net, theta


@pytest.mark.parametrize("g,levels,c0,B", [(8, 1, 8, 1), (8, 1, 40, 3), (16, 2, 24, 1), (32, 1, 8, 2), (32, 3, 16, 1),
                                           (64, 1, 8, 1)])
def test_gradient(g, levels, c0, B):
    print("net gradient: g=%d levels=%d channels=%d batch=%d" % (g, levels, c0, B), flush=True)
    net, theta = _net(g, levels, c0, B, 11)
    rho, T = _inputs(g, B, 5)
    T = U.center(T, U.weights(rho, bf16=True))
    _, grad = net.loss_grad(rho.reshape(B, -1), T.reshape(B, -1, 18))
    _, ref = U.loss_and_grad(theta.astype(np.float64), rho, U.bf16_round(T), levels, c0, bf16=True)
    o = 0
    for name, ci, co, t, _ in U.layer_specs(levels, c0):
        size = co * t * ci + co
        a, b = grad[o:o + size].astype(np.float64), ref[o:o + size]
        o += size
        rel = np.linalg.norm(a - b) / np.linalg.norm(b)
        cos = float(a @ b) / (np.linalg.norm(a) * np.linalg.norm(b))
        print("  %-8s rel L2 %.3e cos %.6f" % (name, rel, cos), flush=True)
        assert rel < 5e-2 and cos > 0.998, name


def test_gradient_is_translation_invariant():
    """Two tiles a row: a rolled sample has the same gradient, but for sums in another order (FP32 over 2^21
    voxels, below 1e-4) and the bf16 roundings of the loss gradient that its weighted mean's last bits move."""
    g, c0 = 128, 8
    print("net gradient, rolled: g=%d" % g, flush=True)
    net, _ = _net(g, 1, c0, 1, 13)
    rho, T = _inputs(g, 1, 7)
    T = U.center(T, U.weights(rho, bf16=True))
    _, a = net.loss_grad(rho.reshape(1, -1), T.reshape(1, -1, 18))
    s = (40, 25, 13)
    _, b = net.loss_grad(np.roll(rho, s, (1, 2, 3)).reshape(1, -1), np.roll(T, s, (1, 2, 3)).reshape(1, -1, 18))
    assert np.linalg.norm(a.astype(np.float64) - b) < 1e-3 * np.linalg.norm(a)
