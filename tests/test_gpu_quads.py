"""Traversal with four lanes per ray: launches whose rays all run that way (the
default below a ray count per class), and the hand-over of a wave's last rays
to it in the larger and in the explicitly configured launches. The reference is
the CPU oracle on the exported tree or the counted one-lane traversal; every
value is computed by the same expressions in all of them, so IDs and bits are
equal."""
import numpy as np
import pytest

from conftest import hit_buffers, to_dev

pytestmark = pytest.mark.gpu
KEYS = ("t", "prim_id", "u", "v")


def _bits(x):
    x = np.asarray(x)
    return x.view(np.uint32) if x.dtype == np.float32 else x


def _rays(n, seed, flat=0.0):
    """Rays into [-1, 1]^3, a share of them along an axis from a grid (their
    origins lie on box planes), some with short intervals."""
    rng = np.random.default_rng(seed)
    r = np.zeros((8, n), np.float32)
    d = rng.normal(size=(3, n))
    r[0:3] = rng.uniform(-1.2, 1.2, (3, n))
    r[3:6] = d / np.linalg.norm(d, axis=0)
    f = rng.random(n) < flat
    r[0:3, f] = 0.25 * rng.integers(-4, 5, (3, int(f.sum())))
    r[3:6, f] = 0.0
    r[3 + rng.integers(0, 3, int(f.sum())), np.flatnonzero(f)] = rng.choice([-1.0, 1.0], int(f.sum()))
    r[7] = np.where(rng.random(n) < 0.2, rng.uniform(0.05, 1.0, n), 1e30)
    return r


def _soup(nt, seed, size=0.08, grid=False):
    rng = np.random.default_rng(seed)
    t = rng.uniform(-1, 1, (nt, 1, 3)) + rng.normal(scale=size, size=(nt, 3, 3))
    if grid:
        t = np.round(t * 4) / 4                       # coincident and degenerate triangles, ties in t
    return t.astype(np.float32).reshape(nt, 9)


def _closest(b, rays, dev, counted=False, **kw):
    import torch
    n = rays.shape[1]
    R, H = to_dev(rays, dev), hit_buffers(n + 64, dev)
    for h in H.values():
        h.fill_(-3)
    out = [H[k][:n] for k in KEYS]
    if counted:
        c = [torch.empty(n, dtype=torch.int32, device=dev) for _ in range(2)]
        b.trace_closest_counted(R, *out, *c)
    else:
        b.trace_closest(R, *out, **kw)
    torch.cuda.synchronize()
    got = {k: H[k].cpu().numpy() for k in KEYS}
    assert all((got[k][n:] == -3).all() for k in KEYS)
    return {k: got[k][:n] for k in KEYS}


def _any(b, rays, dev, counted=False):
    import torch
    n = rays.shape[1]
    occ = torch.full((n + 64,), 7, dtype=torch.uint8, device=dev)
    if counted:
        c = [torch.empty(n, dtype=torch.int32, device=dev) for _ in range(2)]
        b.trace_any_counted(to_dev(rays, dev), occ[:n], *c)
    else:
        b.trace_any(to_dev(rays, dev), occ[:n])
    torch.cuda.synchronize()
    occ = occ.cpu().numpy()
    assert (occ[n:] == 7).all()
    return occ[:n]


def _same(a, b):
    for k in KEYS:
        assert np.array_equal(_bits(a[k]), _bits(b[k])), (k, int((_bits(a[k]) != _bits(b[k])).sum()))


@pytest.mark.parametrize("nt,grid", [(1, False), (3, False), (40, True), (20000, False)])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 64, 65, 3001])
def test_small_launches(pkg, oracle, dev, n, nt, grid):
    """Ray counts at and beside a wave's 16 rays, trees from one leaf up,
    flat rays mixed in; closest hits and occlusion as the oracle's, with the
    borrowed scratch too, and through every configured schedule."""
    rays = _rays(n, 5 * n + nt, flat=0.3)
    with pkg.BVH.build(_soup(nt, nt, size=0.4 if nt < 100 else 0.08, grid=grid)) as b:
        nodes, lt, pid = b.node_data(), np.ascontiguousarray(b.tri_data().T), b.leaf_prim_ids()
        r = oracle.trace_closest(nodes, lt, pid, rays)
        ref = {"t": r["t"], "prim_id": r["id"], "u": r["u"], "v": r["v"]}
        occ = oracle.trace_any(nodes, lt, pid, rays)["occ"]
        _same(_closest(b, rays, dev), ref)
        assert np.array_equal(_any(b, rays, dev), occ)
        H = hit_buffers(n, dev)
        b.trace_closest_no_alloc(to_dev(rays, dev), *[H[k] for k in KEYS])
        import torch
        torch.cuda.synchronize()
        _same({k: H[k].cpu().numpy() for k in KEYS}, ref)
        for sched in (pkg.SCHEDULE_BATCH, pkg.SCHEDULE_REFILL):
            b.set_trace_config(pkg.CLASS_INCOHERENT, sched, 4, 1)
            b.set_trace_config(pkg.CLASS_ANY, sched, 4, 1)
            _same(_closest(b, rays, dev), ref)
            assert np.array_equal(_any(b, rays, dev), occ)


@pytest.mark.parametrize("depth", [4, 8])
def test_deep_tree(pkg, dev, depth):
    """A tree whose stacks pass both LDS depths: triangles in nested shells of
    geometrically shrinking size, so that boxes nest and few rays skip any."""
    rng = np.random.default_rng(3)
    k = np.arange(6000)
    s = (0.5 ** (k / 150.0))[:, None, None]
    tris = (s * rng.normal(size=(6000, 3, 3))).astype(np.float32).reshape(-1, 9)
    rays = _rays(3000, 11)
    rays[0:3] *= rng.uniform(0.0, 1.0, 3000).astype(np.float32) ** 8
    with pkg.BVH.build(tris) as b:
        assert 3 * b.depth + 4 > 24
        ref, occ = _closest(b, rays, dev, counted=True), _any(b, rays, dev, counted=True)
        _same(_closest(b, rays, dev), ref)
        assert np.array_equal(_any(b, rays, dev), occ)
        for sched in (pkg.SCHEDULE_BATCH, pkg.SCHEDULE_REFILL):
            b.set_trace_config(pkg.CLASS_INCOHERENT, sched, depth, 1)
            b.set_trace_config(pkg.CLASS_ANY, sched, depth, 1)
            _same(_closest(b, rays, dev), ref)
            assert np.array_equal(_any(b, rays, dev), occ)
        assert b.trace_status() == 0


@pytest.mark.parametrize("n", [9 << 15, (9 << 15) + 1, 25 << 14, (25 << 14) + 1, 9 << 16, (9 << 16) + 17])
def test_both_sides_of_the_ray_count_rule(pkg, dev, n):
    """Launches at, and just past, the ray counts where the kernels change; a
    queue of the same capacity holding fewer rays."""
    import torch
    rays = _rays(n, n, flat=0.02)
    with pkg.BVH.build(_soup(30000, 8, size=0.03)) as b:
        ref, occ = _closest(b, rays, dev, counted=True), _any(b, rays, dev, counted=True)
        _same(_closest(b, rays, dev), ref)
        assert np.array_equal(_any(b, rays, dev), occ)
        m = n // 3 + 5
        cnt = torch.tensor([m], dtype=torch.int32, device=dev)
        R, H = to_dev(rays, dev), hit_buffers(n, dev)
        for h in H.values():
            h.fill_(-3)
        o = torch.full((n,), 7, dtype=torch.uint8, device=dev)
        b.trace_closest_queued(n, cnt, R, *[H[k] for k in KEYS])
        b.trace_any_queued(n, cnt, R, o)
        torch.cuda.synchronize()
        _same({k: H[k][:m].cpu().numpy() for k in KEYS}, {k: ref[k][:m] for k in KEYS})
        assert all((H[k][m:] == -3).all().item() for k in KEYS)
        assert np.array_equal(o[:m].cpu().numpy(), occ[:m]) and (o[m:] == 7).all().item()


@pytest.mark.parametrize("W,H", [(1, 1), (3, 5), (4, 4), (61, 33), (848, 851), (1025, 1025)])
def test_pinhole_images(pkg, oracle, scenes, dev, W, H):
    """4 x 4 pixel tiles cut off at the right and bottom edge, and an image
    past the ray counts where the batch kernel takes over (848 x 851 in cost
    order, 1025 x 1025 also in plain order): every pixel as the explicit rays' counted trace."""
    import torch
    cam = scenes.parity_camera(W, H)
    rays = oracle.gen_pinhole(scenes.cam_array(cam), W, H)
    c = pkg.camera(cam["o"], cam["f"], cam["r"], cam["u"], cam["scale_x"], cam["scale_y"])
    with pkg.BVH.build(scenes.random_triangles(20000, seed=2)) as b:
        ref = _closest(b, rays, dev, counted=True)
        for flags in (0, pkg.FLAG_COST_ORDER, pkg.FLAG_COST_ORDER):
            hb = hit_buffers(W * H + 64, dev)
            for h in hb.values():
                h.fill_(-3)
            b.trace_pinhole_closest(W, H, c, *[hb[k] for k in KEYS], flags=flags)
            torch.cuda.synchronize()
            got = {k: hb[k].cpu().numpy() for k in KEYS}
            _same({k: got[k][:W * H] for k in KEYS}, ref)
            assert all((got[k][W * H:] == -3).all() for k in KEYS)


KEYS2 = ("t", "inst", "prim_id", "u", "v")


@pytest.fixture(scope="module")
def two_level(pkg, dev):
    """Three meshes (one of a single triangle) in 40 instances: rotated, scaled,
    mirrored, axis-aligned ones, and pairs of the same transform (ties in t,
    decided by the instance)."""
    rng = np.random.default_rng(12)
    meshes = [_soup(4000, 1), _soup(1, 2, size=0.5), _soup(60, 3, size=0.4, grid=True)]
    blas = [pkg.BVH.build(m) for m in meshes]
    o2w = np.zeros((40, 3, 4), np.float32)
    for k in range(40):
        q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
        m = np.eye(3) if k % 4 == 0 else q * rng.uniform(0.3, 1.0) * (1 if k % 3 else -1)
        o2w[k, :, :3], o2w[k, :, 3] = m, rng.uniform(-0.5, 0.5, 3)
    o2w[21:31] = o2w[1:11]
    of = [k % 3 if k < 20 else (k - 20) % 3 for k in range(40)]
    s = pkg.Scene(blas, o2w.reshape(40, 12), of)
    yield s
    s.destroy()
    for b in blas:
        b.destroy()


@pytest.mark.parametrize("n", [1, 15, 16, 17, 64, 65, 3001, 200000])
def test_two_level(pkg, two_level, dev, n):
    """Ray counts at and beside a wave's 16 rays, launches whose rays all start
    in quads and one whose last rays of each wave do, at every stack depth, and
    queues of one ray less; against the counted traversal."""
    import torch
    s, rays = two_level, _rays(n, 3 * n + 1, flat=0.2)
    R = to_dev(rays, dev)

    def buffers():
        f = {k: torch.full((n + 64,), -3, dtype=torch.int32 if k in ("inst", "prim_id") else torch.float32, device=dev)
             for k in KEYS2}
        return f, torch.full((n + 64,), 7, dtype=torch.uint8, device=dev)

    def check(f, occ, m):
        torch.cuda.synchronize()
        for k in KEYS2:
            got = f[k].cpu().numpy()
            assert np.array_equal(_bits(got[:m]), _bits(ref[k][:m])) and (got[m:] == -3).all(), k
        got = occ.cpu().numpy()
        assert np.array_equal(got[:m], hit[:m]) and (got[m:] == 7).all()

    f, _ = buffers()
    c = [torch.empty(n, dtype=torch.int32, device=dev) for _ in range(2)]
    s.trace_closest_counted(R, *[f[k][:n] for k in KEYS2], *c)
    torch.cuda.synchronize()
    ref = {k: f[k][:n].cpu().numpy() for k in KEYS2}
    hit = (ref["prim_id"] >= 0).astype(np.uint8)
    cnt = torch.tensor([n - 1], dtype=torch.int32, device=dev)
    saved = [s.trace_config(k) for k in (0, 1)]
    for depth in (None, 4, 8, 12, 16):
        if depth:
            s.set_trace_config(0, 1, depth, 1)
            s.set_trace_config(1, 2 if depth == 8 else 1, depth, 1)
        f, occ = buffers()
        s.trace_closest(R, *[f[k][:n] for k in KEYS2])
        s.trace_any(R, occ[:n])
        check(f, occ, n)
        f, occ = buffers()
        s.trace_closest_queued(n, cnt, R, *[f[k][:n] for k in KEYS2])
        s.trace_any_queued(n, cnt, R, occ[:n])
        check(f, occ, n - 1)
    for k in (0, 1):
        s.set_trace_config(k, *saved[k])
    assert s.trace_status() == 0
