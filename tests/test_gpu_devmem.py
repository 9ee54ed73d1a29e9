"""The cache of freed device blocks: builds from recycled memory equal the
oracle's (stale contents must not leak in, sizes going up and down, several
handles alive), and cudaBVH_resetDevice gives the cached blocks back."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_recycled_builds_match_oracle(pkg, oracle, scenes, dev):
    kept = []
    for k, n in enumerate((60000, 3000, 60000, 41000, 2049, 65536)):
        print(f"recycled build {n}", flush=True)
        tris = scenes.random_triangles(n, seed=100 + k)
        ob = oracle.OracleBVH(tris)
        b = pkg.BVH.build(tris)
        assert np.array_equal(b.node_data(), ob.nodes())
        assert np.array_equal(b.leaf_prim_ids(), ob.order())
        if k % 2:
            kept.append((b, ob))
        else:
            b.destroy()
    for b, ob in kept:                            # later builds left the earlier handles alone
        assert np.array_equal(b.tri_data().T, ob.leaf_tris())
        b.destroy()


def test_reset_device_returns_the_cache(pkg, scenes, dev):
    import torch
    lib = pkg.load_library()
    tris = scenes.terrain_scene(res=512, spheres=0)
    lib.cudaBVH_resetDevice()
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    for _ in range(3):
        pkg.BVH.build(tris).destroy()
    assert before - torch.cuda.mem_get_info()[0] <= (1 << 30) + (64 << 20)      # bounded while cached
    lib.cudaBVH_resetDevice()
    assert before - torch.cuda.mem_get_info()[0] <= 64 << 20
