"""Compaction of the secondary rays at the edges of its 512-slot tiles and past
the 4,096 tiles that one step of their scan takes: every hit pixel once, in
pixel order, and nothing past the count."""
import numpy as np
import pytest

from conftest import RAY_KEYS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(1, 1), (511, 1), (512, 1), (513, 1), (64, 40), (2048, 1025)])
@pytest.mark.parametrize("share", [0.0, 0.6, 1.0])
def test_compaction(pkg, scenes, dev, W, H, share):
    import torch
    n = W * H
    rng = np.random.default_rng(n)
    hit = rng.random(n) < share
    ids = np.where(hit, rng.integers(0, 500, n), -1).astype(np.int32)
    cam = scenes.parity_camera(W, H)
    c = pkg.camera(cam["o"], cam["f"], cam["r"], cam["u"], cam["scale_x"], cam["scale_y"])
    with pkg.BVH.build(scenes.random_triangles(500, seed=1)) as b:
        t = torch.full((n,), 1.5, device=dev)
        D = {k: torch.full((n,), -7.0, device=dev) for k in RAY_KEYS}
        S = {k: torch.full((n,), -7.0, device=dev) for k in RAY_KEYS}
        src = torch.full((n,), -1, dtype=torch.int32, device=dev)
        cnt = torch.full((1,), -1, dtype=torch.int32, device=dev)
        b.gen_bounce_rays(W, H, c, t, torch.from_numpy(ids).to(dev), 9, (0.0, 4.0, 0.0), D, S, src, cnt)
        torch.cuda.synchronize()
        m = int(hit.sum())
        assert int(cnt.item()) == m
        src = src.cpu().numpy()
        assert np.array_equal(src[:m], np.flatnonzero(hit)) and (src[m:] == -1).all()
        for a in (D, S):
            tmin = a["tmin"].cpu().numpy()
            assert (tmin[:m] == np.float32(1e-3)).all() and (tmin[m:] == -7.0).all()
