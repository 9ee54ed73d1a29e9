"""Handles destroyed while other work goes on: beside a stream capture in relaxed
mode, and while a queued trace on another stream still reads the arrays."""
import numpy as np
import pytest

from conftest import hit_buffers, to_dev

pytestmark = pytest.mark.gpu


def test_destroy_beside_a_relaxed_capture(pkg, scenes, dev):
    """Destroying a handle that has a stream of its own leaves the capture alone."""
    import torch
    own, side = torch.cuda.Stream(), torch.cuda.Stream()
    tris = scenes.random_triangles(60000, seed=1)
    b = pkg.BVH.build(tris)
    b.set_stream(own.cuda_stream)
    x = torch.zeros(1000, device=dev)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side, capture_error_mode="relaxed"):
        x.add_(1.0)
        b.destroy()
        x.mul_(2.0)
    for k in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert (x == 2.0 ** (k + 2) - 2.0).all()
    with pkg.BVH.build(tris) as c:
        assert c.num_tris == 60000


def test_rebuild_after_a_queued_trace(pkg, scenes, dev):
    """A trace is still queued behind long work on its stream when its BVH goes
    and another one of the same size is built: the trace reads the first."""
    import torch
    n = 100000
    rng = np.random.default_rng(2)
    rays = np.zeros((8, n), np.float32)
    rays[0:3] = rng.uniform(-1, 1, (3, n))
    d = rng.normal(size=(3, n))
    rays[3:6] = d / np.linalg.norm(d, axis=0)
    rays[7] = 1e30
    R = to_dev(rays, dev)
    first, second = scenes.random_triangles(60000, seed=3), scenes.random_triangles(60000, seed=4)
    with pkg.BVH.build(first) as b:
        H = hit_buffers(n, dev)
        b.trace_closest(R, H["t"], H["prim_id"], H["u"], H["v"])
        torch.cuda.synchronize()
        ref = H["t"].clone()
    s = torch.cuda.Stream()
    for _ in range(3):
        b = pkg.BVH.build(first)
        b.set_stream(s.cuda_stream)
        H = hit_buffers(n, dev)
        b.trace_closest(R, H["t"], H["prim_id"], H["u"], H["v"])        # its scratch
        torch.cuda.synchronize()
        H["t"].fill_(-1.0)
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            torch.cuda._sleep(20_000_000)
        b.trace_closest(R, H["t"], H["prim_id"], H["u"], H["v"])
        b.set_stream(None)                      # the last trace is on a stream that is no longer the handle's
        b.destroy()
        c = pkg.BVH.build(second)
        torch.cuda.synchronize()
        assert torch.equal(H["t"], ref)
        c.destroy()
