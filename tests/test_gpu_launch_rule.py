"""Which kernel a small launch takes follows the class's configuration: four lanes
per ray (64-thread workgroups) with the default one, the configured schedule
(256-thread workgroups) with any other, whether it was set or found by the
autotuner."""
import numpy as np
import pytest

from conftest import hit_buffers, to_dev

pytestmark = pytest.mark.gpu
DEFAULT = (3, 8, 0)


def _rays(n, dev):
    rng = np.random.default_rng(n)
    r = np.zeros((8, n), np.float32)
    r[0:3] = rng.uniform(-1, 1, (3, n))
    d = rng.normal(size=(3, n))
    r[3:6] = d / np.linalg.norm(d, axis=0)
    r[7] = 1e30
    return to_dev(r, dev)


@pytest.fixture()
def bvh(pkg, scenes, dev):
    with pkg.BVH.build(scenes.random_triangles(5000, seed=1)) as b:
        yield b


@pytest.fixture()
def threads(pkg, bvh, dev):
    R, H = _rays(3000, dev), hit_buffers(3000, dev)

    def run():
        import torch
        bvh.trace_closest(R, H["t"], H["prim_id"], H["u"], H["v"])
        torch.cuda.synchronize()
        return bvh.launch_info()["threads_per_workgroup"]
    return run


def test_set_and_restore(pkg, bvh, threads):
    cls = pkg.CLASS_INCOHERENT
    assert bvh.trace_config(cls) == DEFAULT and threads() == 64
    bvh.set_trace_config(cls, *bvh.trace_config(cls))
    assert threads() == 64
    bvh.set_trace_config(cls, 0, 12, 0)
    assert threads() == 256
    bvh.set_trace_config(cls, *bvh.trace_config(cls))
    assert threads() == 256
    bvh.set_trace_config(cls, *DEFAULT)
    assert threads() == 64


def test_autotune_on_a_small_workload(pkg, bvh, threads, dev):
    """What the autotuner keeps is what runs. The default one, four lanes per
    ray there, is a candidate; started from another configuration too."""
    cls = pkg.CLASS_INCOHERENT
    for first in (None, (1, 16, 0)):
        if first:
            bvh.set_trace_config(cls, *first)
        best, table = bvh.autotune(cls, reps=2, rays=_rays(3000, dev))
        assert bvh.trace_config(cls) == best and len(table) == 36
        assert best == min(table, key=lambda r: r[3])[:3]
        assert threads() == (64 if best == DEFAULT else 256)


def test_autotune_on_a_large_workload(pkg, bvh, threads, dev):
    """More rays than would get four lanes each: small launches stay as they were."""
    cls = pkg.CLASS_INCOHERENT
    big = _rays((9 << 15) + 1, dev)
    best, _ = bvh.autotune(cls, reps=1, rays=big)
    assert threads() == 64
    bvh.set_trace_config(cls, *best)
    assert threads() == 64
    bvh.set_trace_config(cls, *DEFAULT)
    bvh.set_trace_config(cls, 0, 16, 0)
    bvh.autotune(cls, reps=1, rays=big)
    assert threads() == 256


@pytest.mark.parametrize("n", [1, 3000, 100000])
def test_launch_info_of_small_launches(pkg, bvh, dev, n):
    """Workgroups and waves as many as the rays take, up to what fits."""
    import torch
    R, H = _rays(n, dev), hit_buffers(n, dev)
    bvh.trace_closest(R, H["t"], H["prim_id"], H["u"], H["v"])
    torch.cuda.synchronize()
    info = bvh.launch_info()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert info["threads_per_workgroup"] == 64 and info["workgroups"] == (n + 15) // 16
    assert info["blocks_per_cu"] == min(info["max_blocks_per_cu"], -(-info["workgroups"] // cus))
    assert info["waves_per_simd"] == -(-info["blocks_per_cu"] // 4)
