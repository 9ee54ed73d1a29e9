"""Bounds of every tree of a set built in one pass: those of a sequential pass over
its own triangles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bounds(t):
    p = t.reshape(-1, 3)
    mn, mx = np.full(3, 1e30, np.float32), np.full(3, -1e30, np.float32)
    for v in p:                                    # the first of equal values, NaN skipped
        mn, mx = np.where(v < mn, v, mn), np.where(mx < v, v, mx)
    e = (mx - mn).astype(np.float32)
    ext = np.sqrt(np.float32(np.float32(e[0] * e[0] + e[1] * e[1]) + e[2] * e[2]))
    return tuple(((mn + mx) * np.float32(0.5)).tolist()) + (float(ext),)


@pytest.mark.parametrize("counts", [[1, 4, 5, 100], [5, 6, 2048, 2049, 4096, 4097, 3], [4100] * 3 + [7] * 40])
def test_bounds_of_each_tree(pkg, scenes, dev, counts):
    import torch
    rng = np.random.default_rng(len(counts))
    tris = []
    for k, n in enumerate(counts):
        t = (scenes.random_triangles(n, seed=k).reshape(-1, 9) * np.float32(1 + k) + np.float32(k)).astype(np.float32)
        if k % 3 == 1:                             # flat on one side, zeros of both signs
            t = np.abs(t)
            t[:, 1::3] = np.where(rng.random((n, 3)) < 0.5, np.float32(0.0), np.float32(-0.0))
        tris.append(t)
    vs = [torch.from_numpy(t).to(dev).reshape(-1) for t in tris]
    built = pkg.BVH.build_many_device([[(v, None, 12, v.numel() // 3, v.numel() // 9)] for v in vs])
    for t, b in zip(tris, built):
        want = np.asarray(_bounds(t), np.float32)
        assert np.array_equal(np.asarray(b.bounds(), np.float32).view(np.uint32), want.view(np.uint32))
        with pkg.BVH.build(t) as own:
            assert own.bounds() == b.bounds()
        b.destroy()
    big = [t for t in tris if len(t) > 4]
    batch = pkg.Batch(big)
    want = np.asarray(_bounds(np.concatenate(big)), np.float32)
    assert np.array_equal(np.asarray(batch.forest().bounds(), np.float32).view(np.uint32), want.view(np.uint32))
    batch.destroy()
