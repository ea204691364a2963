"""The convolution kernels where their tiles end: image widths off the 16- and
32-pixel tiles or equal to one, levels of a single pixel, channel counts off the
32-channel K step and the output tiles, and pixels too wide for LDS."""
import numpy as np
import pytest

import test_gpu_net as base
from oracle import net_oracle as no

pytestmark = pytest.mark.gpu

SHAPES = [(8, 8, (8, 8, 8, 8), 1), (8, 96, (8, 16, 24, 48), 2), (32, 64, (32, 64, 80, 112), 1),
          (24, 160, (16, 32, 56, 104), 2), (16, 16, (376, 376, 376, 384), 2)]


@pytest.mark.parametrize("H,W,widths,B", SHAPES)
def test_forward_is_exact(hip, H, W, widths, B):
    """Sums of at most two short dyadic terms: no order and no rounding differ."""
    from lbm_mirror_amd.warmstart import Net
    rng = np.random.default_rng(31)
    net = Net(H, W, widths, batch=B, seed=12)
    net.set_params(base._dyadic_params(widths, rng))
    x = no.bf16(base._x(rng, B, H, W))
    assert np.array_equal(net.forward_raw(x), no.forward(net.get_params(), widths, x, mode="bf16"))


@pytest.mark.parametrize("H,W,widths,B", SHAPES)
def test_gradient_with_exact_arithmetic(hip, H, W, widths, B):
    """Every gradient tensor where only its own FP32 sum over pixels rounds."""
    from lbm_mirror_amd.warmstart import Net
    rng = np.random.default_rng(23)
    net = Net(H, W, widths, batch=B, seed=12)
    net.set_params(base._dyadic_params(widths, rng))
    params = net.get_params()
    x = no.bf16(base._x(rng, B, H, W))
    ref = no.forward(params, widths, x, mode="bf16")
    t = (ref + rng.choice([-0.5, -0.25, 0.25, 0.5], ref.shape)).astype(np.float32)
    m = np.zeros(B * H * W, np.float32)
    m[rng.permutation(B * H * W)[: 1 << int(np.log2(B * H * W // 2))]] = 1
    m = m.reshape(B, H, W)
    loss, g = net.loss_grad_raw(x, t, m)
    lref, gref = no.loss_grad(params, widths, x, t, m, mode="bf16")
    assert abs(loss - lref) <= 1e-9 * lref
    off = 0
    for i, (ci, co, _, _) in enumerate(no.layer_specs(widths)):
        for n in (9 * ci * co, co):
            err = np.linalg.norm(g[off:off + n] - gref[off:off + n])
            assert err <= 1e-5 * np.linalg.norm(gref[off:off + n]), (i, n, err)
            off += n
