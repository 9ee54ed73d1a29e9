"""Closest hits where many triangles are hit at equal t and many boxes are entered
at equal distances: axis-aligned floors cut into a grid, with rays aimed at shared
vertices, and triangles on a coarse grid. A box's entry distance can round above a
hit's t there, so the answer depends on the order in which boxes are visited and
on which triangles of a leaf are tested; it has to be the one-lane traversal's
(the counted launches') in every launch."""
import numpy as np
import pytest

from conftest import hit_buffers, to_dev

pytestmark = pytest.mark.gpu
KEYS = ("t", "prim_id", "u", "v")
KEYS2 = ("t", "inst", "prim_id", "u", "v")


def _floors(n=48):
    g = np.linspace(-1, 1, n + 1, dtype=np.float32)
    x, z = [a.ravel() for a in np.meshgrid(g[:-1], g[:-1], indexing="ij")]
    X, Z = [a.ravel() for a in np.meshgrid(g[1:], g[1:], indexing="ij")]
    tris = []
    for y in (-0.5, 0.0, 0.25):
        y = np.full_like(x, y)
        tris.append(np.stack([x, y, z, X, y, z, X, y, Z], 1))
        tris.append(np.stack([x, y, z, X, y, Z, x, y, Z], 1))
    return np.concatenate(tris).astype(np.float32)


def _grid_soup(nt=20000):
    rng = np.random.default_rng(4)
    t = rng.uniform(-1, 1, (nt, 1, 3)) + rng.normal(scale=0.2, size=(nt, 3, 3))
    return (np.round(t * 4) / 4).astype(np.float32).reshape(nt, 9)


def _rays(n, tris, seed):
    """Seven in ten aimed at a vertex, the others in random directions."""
    rng = np.random.default_rng(seed)
    r = np.zeros((8, n), np.float32)
    r[0:3] = rng.uniform(-1.2, 1.2, (3, n))
    d = tris.reshape(-1, 3)[rng.integers(0, 3 * len(tris), n)].T - r[0:3]
    d = np.where(rng.random(n) < 0.3, rng.normal(size=(3, n)), d)
    r[3:6] = d / np.maximum(np.linalg.norm(d, axis=0), 1e-6)
    r[7] = 1e30
    return r


def _out(keys, n, dev):
    import torch
    return [torch.full((n,), -3, dtype=torch.int32 if k in ("inst", "prim_id") else torch.float32, device=dev)
            for k in keys]


def _differing(a, b):
    import torch
    torch.cuda.synchronize()
    return {i: int((x != y).sum()) for i, (x, y) in enumerate(zip(a, b)) if (x != y).any()}


def _counted(s, R, keys, n, dev):
    import torch
    ref, c = _out(keys, n, dev), [torch.empty(n, dtype=torch.int32, device=dev) for _ in range(2)]
    s.trace_closest_counted(R, *ref, *c)
    return ref


@pytest.fixture(scope="module", params=["floors", "grid_soup"])
def mesh(request, pkg, dev):
    tris = _floors() if request.param == "floors" else _grid_soup()
    with pkg.BVH.build(tris) as b:
        yield tris, b


@pytest.fixture(scope="module")
def scene(mesh, pkg):
    """Sixteen instances moved by and scaled to powers of two, some of them twice."""
    tris, b = mesh
    rng = np.random.default_rng(6)
    m = np.zeros((16, 3, 4), np.float32)
    s = 2.0 ** rng.integers(-2, 1, 16)
    for a in range(3):
        m[:, a, a] = s
    m[:, :, 3] = rng.integers(-2, 3, (16, 3)) / 4
    m[12:] = m[:4]
    s = pkg.Scene([b], m.reshape(16, 12), [0] * 16)
    pts = np.einsum("kij,pj->kpi", m[:, :, :3], tris.reshape(-1, 3)[:3000]) + m[:, None, :, 3]
    yield pts.astype(np.float32).reshape(-1, 9), s
    s.destroy()


@pytest.mark.parametrize("n", [4000, 200000])
def test_four_lanes_per_ray_from_the_root(mesh, dev, n):
    tris, b = mesh
    R = to_dev(_rays(n, tris, n), dev)
    got = _out(KEYS, n, dev)
    b.trace_closest(R, *got)
    assert _differing(got, _counted(b, R, KEYS, n, dev)) == {}


@pytest.mark.parametrize("n", [4000, 60000])
def test_two_level_four_lanes_per_ray_from_the_root(scene, dev, n):
    pts, s = scene
    R = to_dev(_rays(n, pts, n), dev)
    got = _out(KEYS2, n, dev)
    s.trace_closest(R, *got)
    assert _differing(got, _counted(s, R, KEYS2, n, dev)) == {}


@pytest.mark.parametrize("config", [(0, 8, 0), (0, 12, 2), (3, 8, 2), (3, 12, 0)])
@pytest.mark.parametrize("n", [200000, 1000000])
def test_hand_over_within_a_leaf(mesh, pkg, dev, config, n):
    """A wave's last rays change to four lanes each wherever they are: also
    between two triangles of a leaf, all of which are still to be tested."""
    tris, b = mesh
    R = to_dev(_rays(n, tris, n + 1), dev)
    ref = _counted(b, R, KEYS, n, dev)
    saved = b.trace_config(pkg.CLASS_INCOHERENT)
    b.set_trace_config(pkg.CLASS_INCOHERENT, *config)
    got = _out(KEYS, n, dev)
    b.trace_closest(R, *got)
    b.set_trace_config(pkg.CLASS_INCOHERENT, *saved)
    assert _differing(got, ref) == {}


@pytest.mark.parametrize("n", [200000, 600000])
def test_two_level_hand_over_within_a_leaf(scene, dev, n):
    pts, s = scene
    R = to_dev(_rays(n, pts, n + 1), dev)
    got = _out(KEYS2, n, dev)
    s.trace_closest(R, *got)
    assert _differing(got, _counted(s, R, KEYS2, n, dev)) == {}
