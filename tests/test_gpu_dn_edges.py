"""Weight gradients of the first layer where one input is NaN: exactly the taps that
bring that pixel to a pixel of the image are NaN, also beside the edges of the
kernel's tiles and of the image."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(8, 8), (24, 16), (32, 8), (40, 24), (72, 8)])
def test_nan_input_reaches_its_own_taps(pkg, dev, W, H):
    import torch
    rng = np.random.default_rng(W + H)
    x = torch.from_numpy(rng.normal(size=(H, W, 16)).astype(np.float32)).to(dev).bfloat16()
    target = torch.from_numpy(rng.gamma(1.0, 1.0, 3 * W * H).astype(np.float32)).to(dev)
    for px, py in ((0, 0), (W - 1, 0), (0, H - 1), (W - 1, H - 1), (W // 2, H // 2), (min(31, W - 1), 3)):
        d = pkg.Denoiser(4096, seed=1)
        y = x.clone()
        y[py, px, 5] = float("nan")
        d.train_step(1, H, W, y.view(torch.int16).reshape(-1), target, 1e-3)
        g = d.params(1)
        d.destroy()
        want = np.zeros((32, 9, 16), bool)
        for t in range(9):
            qx, qy = px - (t % 3 - 1), py - (t // 3 - 1)        # the output pixel whose tap t reads (px, py)
            want[:, t, 5] = 0 <= qx < W and 0 <= qy < H
        assert np.array_equal(np.isnan(g[:want.size]).reshape(want.shape), want), (px, py)
        assert np.isfinite(g[want.size:]).all()
