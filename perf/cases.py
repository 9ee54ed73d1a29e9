"""Timed cases of the framework's use: what each runs, on which inputs, and
the work it cannot do without.

A case is a dict of plain values: `kind` selects what runs, the rest are its
sizes and options. `listed()` names the standing set, `draw(rng)` gives one
more case of the same ranges, `prepare` makes what a program holds before the
call (geometry, handles, weights, buffers), `run` makes one pass through the
public entry points, `work` states its bytes and operations, and `exact` gives
the outputs in 64-bit arithmetic where that is practical.
"""
from __future__ import annotations

import importlib
import math

import numpy as np
import torch

pkg = importlib.import_module("vk-rt-cuda-raytracing_amd")
scenes = importlib.import_module("vk-rt-cuda-raytracing_amd.scenes")
denoise_train = importlib.import_module("vk-rt-cuda-raytracing_amd.denoise_train")

RAY_KEYS = ("ox", "oy", "oz", "dx", "dy", "dz", "tmin", "tmax")
MISS_T = 1e30


def listed():
    return [
        # A picking query or a small probe batch on a small mesh: one launch, latency only.
        dict(name="rays_4k", kind="rays", tris=4096, rays=4096, any_hit=False, sort=False),
        # A preview frame on a mid-size mesh: 512 x 512 primaries on 65,536 random triangles,
        # one diffuse bounce and one shadow ray per hit.
        dict(name="frame_512", kind="frame", scene="soup", tris=65536, width=512, height=512),
        # A full frame on the large static world: 3.4 M triangles, 1920 x 1080 primaries, diffuse
        # bounce and shadow ray per hit.
        dict(name="frame_1080p", kind="frame", scene="terrain", res=1024, spheres=256, width=1920, height=1080),
        # Loading one mesh from host triangles and handing its exports (BVH4 nodes, packed
        # triangles) to a ray-query consumer.
        dict(name="build_64k", kind="build", tris=65536),
        # Geometry that changes on the device: rebuild from vertex / index buffers, then trace a
        # 720p frame of it.
        dict(name="rebuild_3m", kind="rebuild", res=1024, spheres=256, width=1280, height=720, index16=False),
        # An instance update: the top-level structure of 4,096 instance boxes, every frame.
        dict(name="tlas_4k", kind="tlas", boxes=4096),
        # Ray queries into an instanced world: closest hit of camera and scattered rays, any hit
        # of rays toward the sun.
        dict(name="scene_rays_1m", kind="scene_rays", instances=64, rays=1 << 20),
        # Offline or interactive path tracing of the instanced world: 4 samples of a 1080p frame.
        dict(name="path_1080p", kind="path", instances=64, width=1920, height=1080, spp=4, depth=8),
        # Many independent scenes served together: one replayed launch for all their rays.
        dict(name="batch_trace_64", kind="batch_trace", scenes=64, tris_max=200000, rays_max=1 << 20),
        # New scenes arriving together: one forest build, then their first rays (any hit).
        dict(name="batch_build_64", kind="batch_build", scenes=64, tris_max=200000, rays_max=1 << 16),
        # Denoising a rendered 1080p frame.
        dict(name="denoise_1080p", kind="denoise", width=1920, height=1080),
        # One training step of the denoiser on eight 256 x 256 crops, at the learning rate of the
        # end of the cosine schedule (the weights hardly move, so every pass sees the same network).
        dict(name="train_8x256", kind="train", batch=8, size=256),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rays", "frame", "frame", "build", "rebuild", "tlas", "scene_rays", "path", "batch_trace",
                       "batch_build", "denoise", "train"])
    if kind == "rays":
        return dict(kind=kind, tris=_log(rng, 1000, 200000), rays=_log(rng, 1000, 1 << 21),
                    any_hit=rng.random() < 0.4, sort=rng.random() < 0.3)
    if kind == "frame":
        w = _log(rng, 64, 1920)
        h = max(1, min(1080, int(w * rng.uniform(0.5, 1.0))))
        if rng.random() < 0.5:
            return dict(kind=kind, scene="soup", tris=_log(rng, 1000, 200000), width=w, height=h)
        return dict(kind=kind, scene="terrain", res=_log(rng, 64, 1024), spheres=rng.randint(0, 256), width=w, height=h)
    if kind == "build":
        return dict(kind=kind, tris=_log(rng, 1, 1 << 18))
    if kind == "rebuild":
        small = rng.random() < 0.3
        res, spheres = (_log(rng, 4, 200), 0) if small else (_log(rng, 16, 1024), rng.randint(0, 256))
        w = _log(rng, 320, 1280)
        return dict(kind=kind, res=res, spheres=spheres, width=w, height=max(1, int(w * rng.uniform(0.4, 0.56))),
                    index16=small)
    if kind == "tlas":
        return dict(kind=kind, boxes=_log(rng, 1, 100000))
    if kind == "scene_rays":
        return dict(kind=kind, instances=rng.randint(1, 64), rays=_log(rng, 1000, 1 << 20))
    if kind == "path":
        w = _log(rng, 128, 1920)
        return dict(kind=kind, instances=rng.randint(4, 64), width=w, height=max(8, int(w * rng.uniform(0.45, 0.5625))),
                    spp=rng.randint(1, 4), depth=rng.randint(2, 8))
    if kind in ("batch_trace", "batch_build"):
        return dict(kind=kind, scenes=rng.randint(2, 64), tris_max=_log(rng, 5000, 200000),
                    rays_max=_log(rng, 1 << 16, 1 << 20) if kind == "batch_trace" else 1 << 16)
    if kind == "denoise":
        w = 8 * _log(rng, 8, 240)
        return dict(kind=kind, width=w, height=8 * max(1, min(135, int(w * rng.uniform(0.4, 0.5625)) // 8)))
    return dict(kind="train", batch=rng.randint(1, 8), size=8 * _log(rng, 8, 32))


# ----------------------------------------------------------------- inputs ----
def _dev():
    return torch.device("cuda:0")


def _gen(seed):
    g = torch.Generator(device=_dev())
    g.manual_seed(int(seed))
    return g


def _f(*shape):
    return torch.zeros(*shape, device=_dev())


def _i(*shape):
    return torch.zeros(*shape, dtype=torch.int32, device=_dev())


def _cam(c):
    return pkg.camera(c["o"], c["f"], c["r"], c["u"], c["scale_x"], c["scale_y"])


def _terrain_mesh(res, spheres, seed):
    """Vertex (n, 3) float32 and index (m, 3) int32 device buffers of the
    heightfield (res x res cells over [-10, 10]^2, six sine octaves) with
    level-4 icospheres resting on it."""
    dev = _dev()
    rng = np.random.default_rng(seed)
    theta, phase = rng.uniform(0.0, 2.0 * np.pi, 6), rng.uniform(0.0, 2.0 * np.pi, 6)

    def height(x, z):
        return sum(0.5 ** k * torch.sin(0.35 * 2.0 ** k * (x * math.cos(theta[k]) + z * math.sin(theta[k])) + phase[k])
                   for k in range(6))

    g = torch.linspace(-10.0, 10.0, res + 1, device=dev, dtype=torch.float64)
    z, x = torch.meshgrid(g, g, indexing="ij")
    vert = [torch.stack([x, height(x, z), z], -1).reshape(-1, 3).float()]
    c = torch.arange(res, device=dev)
    a = ((c[:, None] * (res + 1)) + c[None]).reshape(-1)
    idx = [torch.stack([torch.stack([a, a + 1, a + res + 2], -1),
                        torch.stack([a, a + res + 2, a + res + 1], -1)], 1).reshape(-1, 3)]
    if spheres > 0:
        unit = torch.from_numpy(scenes.icosphere(4).reshape(-1, 3)).to(dev)       # triangle corners
        r = np.random.default_rng(seed + 1000)
        cx, cz, rad, up = (torch.from_numpy(r.uniform(lo, hi, spheres)).to(dev)
                           for lo, hi in ((-9, 9), (-9, 9), (0.1, 1.0), (0.3, 1.2)))
        cen = torch.stack([cx, height(cx, cz) + rad * up, cz], -1)
        s = (unit[None] * rad[:, None, None] + cen[:, None]).reshape(-1, 3).float()
        idx.append(torch.arange(s.shape[0], device=dev).reshape(-1, 3) + vert[0].shape[0])
        vert.append(s)
    return torch.cat(vert).contiguous(), torch.cat(idx).to(torch.int32).contiguous()


def _soup(n, seed):
    """scenes.random_triangles' distribution, drawn on the device: (n, 9)."""
    g, dev = _gen(seed), _dev()
    c = torch.rand(n, 1, 3, device=dev, generator=g, dtype=torch.float64) * 2 - 1
    d = torch.randn(n, 3, 3, device=dev, generator=g, dtype=torch.float64)
    d = d / d.norm(dim=2, keepdim=True)
    ln = 0.005 + 0.045 * torch.rand(n, 3, 1, device=dev, generator=g, dtype=torch.float64)
    return (c + d * ln).float().reshape(n, 9).contiguous()


def _specs(case):
    return scenes.batch_specs(case["scenes"], tris=(1000, case["tris_max"]),
                              rays=(4096, case["rays_max"]) if case["kind"] == "batch_build" else (65536, case["rays_max"]))


def _planes(w, h, seed, noisy=True):
    """A rendered frame's planes: patches of albedo and normal, smooth
    radiance (with one-sample noise when noisy) and depth; channel-major."""
    g, dev = _gen(seed), _dev()
    y = torch.arange(h, device=dev, dtype=torch.float32)[:, None] / 128.0
    x = torch.arange(w, device=dev, dtype=torch.float32)[None] / 128.0
    ph = torch.rand(8, device=dev, generator=g) * 6.28
    fr = torch.rand(8, device=dev, generator=g) * 3 + 0.5
    bump = sum(torch.sin(fr[k] * x + ph[k]) * torch.cos(fr[k + 4] * y + ph[k + 4]) for k in range(4)) / 4
    cell = ((torch.floor(2 * x + bump) * 131 + torch.floor(2 * y - bump) * 71).long() % 64)
    alb = (0.2 + 0.6 * torch.rand(3, 64, device=dev, generator=g))[:, cell]
    nrm = torch.randn(3, 64, device=dev, generator=g)[:, cell] + torch.stack([bump, 1 - bump, bump * bump])
    nrm = nrm / nrm.norm(dim=0, keepdim=True)
    dep = 6 + 4 * bump + 0.2 * cell.float()
    clean = alb * (1.2 + bump)
    rgb = clean
    if noisy:
        rgb = clean * -torch.log(1 - 0.999 * torch.rand(3, h, w, device=dev, generator=g))
    return tuple(t.reshape(-1).contiguous() for t in (rgb, alb, nrm, dep, clean))


def _train_data(case, seed):
    """BF16 inputs (B, S, S, 16: ten channels used) and log-space targets."""
    S, B = case["size"], case["batch"]
    X = torch.zeros(B, S, S, 16, dtype=torch.bfloat16, device=_dev())
    Y = torch.zeros(B, S, S, 3, device=_dev())
    for b in range(B):
        rgb, alb, nrm, dep, clean = _planes(S, S, seed * 64 + b)
        ch = torch.cat([torch.log1p(rgb), alb, nrm, torch.log1p(dep) * 0.25]).view(10, S, S)
        X[b, :, :, :10] = ch.permute(1, 2, 0).bfloat16()
        Y[b] = torch.log1p(clean).view(3, S, S).permute(1, 2, 0)
    return X, Y


def _query_rays(n, seed):
    """Rays into the instanced world: half camera rays, half from points in it
    in random directions; and shadow rays toward the sun."""
    dev, g = _dev(), _gen(seed)
    k = n // 2
    w = max(1, int(math.sqrt(max(k, 1))))
    cam = scenes.instanced_camera(w, max(1, (k + w - 1) // w))
    i = torch.arange(k, device=dev)
    hh = max(1, (k + w - 1) // w)
    sx = (((i % w).float() + 0.5) / w * 2 - 1) * float(cam["scale_x"])
    sy = (((i // w).float() + 0.5) / hh * 2 - 1) * float(cam["scale_y"])
    f, r, u, o = (torch.tensor(cam[q], device=dev)[:, None] for q in ("f", "r", "u", "o"))
    d1 = f + sx * r + sy * u
    d2 = torch.randn(3, n - k, device=dev, generator=g)
    O = torch.cat([o.expand(3, k), torch.rand(3, n - k, device=dev, generator=g) * 20 - 10], 1)
    D = torch.cat([d1 / d1.norm(dim=0), d2 / d2.norm(dim=0)], 1)
    so = torch.rand(3, n, device=dev, generator=g) * 20 - 10
    sun = torch.tensor(scenes.SUN_DIR, device=dev)
    sd = (sun / sun.norm())[:, None].expand(3, n)
    return _rays(O, D), _rays(so, sd)


def _rays(o, d):
    n = o.shape[1]
    R = {k: o[j].clone() for j, k in enumerate(("ox", "oy", "oz"))}
    R.update({k: d[j].clone() for j, k in enumerate(("dx", "dy", "dz"))})
    R["tmin"], R["tmax"] = _f(n), torch.full((n,), MISS_T, device=_dev())
    return R


def prepare(case, seed):
    kind = case["kind"]
    s = dict(kind=kind, case=case)
    if kind == "rays":
        n = case["rays"]
        v = _soup(case["tris"], seed)
        s["bvh"] = pkg.BVH.build_device(v, case["tris"])
        s["rays"] = _rays(*scenes.batch_rays_device(n, seed + 1, _dev()))
        s["t"], s["id"], s["u"], s["v"] = _f(n), _i(n), _f(n), _f(n)
        s["occ"] = torch.zeros(n, dtype=torch.uint8, device=_dev())
    elif kind == "frame":
        W, H = case["width"], case["height"]
        n = W * H
        if case["scene"] == "soup":
            s["bvh"] = pkg.BVH.build_device(_soup(case["tris"], seed), case["tris"])
            cam, s["light"] = scenes.parity_camera(W, H), (0.0, 4.0, 0.0)
        else:
            v, i = _terrain_mesh(case["res"], case["spheres"], seed)
            s["bvh"] = pkg.BVH.build_device(v, i.shape[0], i)
            cam, s["light"] = scenes.terrain_camera(W, H), scenes.TERRAIN_LIGHT
        s["cam"], s["seed"] = _cam(cam), seed & 0x7fffffff
        s["primary"] = dict(t=_f(n), id=_i(n), u=_f(n), v=_f(n))
        s["D"] = {k: _f(n) for k in RAY_KEYS}
        s["S"] = {k: _f(n) for k in RAY_KEYS}
        s["src"], s["count"] = _i(n), _i(1)
        s["diffuse"] = dict(t=_f(n), id=_i(n), u=_f(n), v=_f(n))
        s["occ"] = torch.zeros(n, dtype=torch.uint8, device=_dev())
    elif kind == "build":
        s["tris"] = _soup(case["tris"], seed).cpu().numpy()
        # the consumer's node buffer, sized for any tree of so many triangles
        s["nodes"] = np.zeros((case["tris"], 64), np.uint8)
    elif kind == "rebuild":
        W, H = case["width"], case["height"]
        s["v"], s["i"] = _terrain_mesh(case["res"], case["spheres"], seed)
        if case["index16"]:
            s["i"] = s["i"].to(torch.int16)
        s["cam"] = _cam(scenes.terrain_camera(W, H))
        n = W * H
        s["t"], s["id"], s["u"], s["v2"] = _f(n), _i(n), _f(n), _f(n)
    elif kind == "tlas":
        rng = np.random.default_rng(seed)
        c = rng.uniform(-10, 10, (case["boxes"], 3))
        e = rng.uniform(0.25, 1.0, (case["boxes"], 3))
        s["aabbs"] = np.concatenate([c - e, c + e], 1).astype(np.float32)
    elif kind in ("scene_rays", "path"):
        sc = scenes.instanced_scene(n_inst=case["instances"], seed=seed & 0xffff)
        s["blas"] = [pkg.BVH.build(m) for m in sc["meshes"]]
        s["scene"] = pkg.Scene(s["blas"], sc["o2w"], sc["blas_of"], sc["albedo"])
        if kind == "scene_rays":
            n = case["rays"]
            s["rays"], s["shadow"] = _query_rays(n, seed)
            s["t"], s["inst"], s["prim"], s["u"], s["v"] = _f(n), _i(n), _i(n), _f(n), _f(n)
            s["occ"] = torch.zeros(n, dtype=torch.uint8, device=_dev())
        else:
            W, H = case["width"], case["height"]
            s["cam"] = _cam(scenes.instanced_camera(W, H))
            s["params"] = pkg.path_params(W, H, spp=case["spp"], max_depth=case["depth"], seed=1 + (seed & 0xffff))
            s["rgb"], s["alb"], s["nrm"], s["dep"] = _f(3 * W * H), _f(3 * W * H), _f(3 * W * H), _f(W * H)
    elif kind in ("batch_trace", "batch_build"):
        specs = _specs(case)
        s["tris"] = [_soup(nt, seed + 1 + k).cpu().numpy() for k, (nt, _) in enumerate(specs)]
        s["rays"], off = scenes.batch_workload_device(specs, _dev(), seed0=seed + 7000)
        n = s["n"] = int(off[-1])
        s["off"] = torch.from_numpy(off).to(_dev())
        if kind == "batch_trace":
            s["batch"] = pkg.Batch(s.pop("tris"))
            s["t"], s["id"], s["u"], s["v"] = _f(n), _i(n), _f(n), _f(n)
        else:
            s["occ"] = torch.zeros(n, dtype=torch.uint8, device=_dev())
    elif kind == "denoise":
        W, H = case["width"], case["height"]
        s["dn"] = pkg.Denoiser((W * H + 63) // 64 * 64, seed=0)
        s["dn"].set_params(denoise_train.load_weights())
        s["planes"] = _planes(W, H, seed)[:4]
        s["out"] = _f(3 * W * H)
    else:
        B, S = case["batch"], case["size"]
        s["dn"] = pkg.Denoiser(B * S * S, seed=0)
        s["dn"].set_params(denoise_train.load_weights())
        s["x"], s["y"] = _train_data(case, seed)
    return s


# -------------------------------------------------------------------- run ----
def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "rays":
        flags = pkg.FLAG_SORT_RAYS if case["sort"] else 0
        if case["any_hit"]:
            s["bvh"].trace_any(s["rays"], s["occ"], flags=flags)
            return s["occ"]
        s["bvh"].trace_closest(s["rays"], s["t"], s["id"], s["u"], s["v"], flags=flags)
        return {k: s[k] for k in ("t", "id", "u", "v")}
    if kind == "frame":
        W, H, b, p, d = case["width"], case["height"], s["bvh"], s["primary"], s["diffuse"]
        b.trace_pinhole_closest(W, H, s["cam"], p["t"], p["id"], p["u"], p["v"], flags=pkg.FLAG_COST_ORDER)
        b.gen_bounce_rays(W, H, s["cam"], p["t"], p["id"], s["seed"], s["light"], s["D"], s["S"], s["src"], s["count"],
                          flags=pkg.FLAG_TILE_ORDER)
        b.trace_closest_queued(W * H, s["count"], s["D"], d["t"], d["id"], d["u"], d["v"])
        b.trace_any_queued(W * H, s["count"], s["S"], s["occ"])
        return {k: s[k] for k in ("primary", "D", "S", "src", "count", "diffuse", "occ")}
    if kind == "build":
        with pkg.BVH.build(s["tris"]) as b:
            nodes = b.node_data()
            s["nodes"][:len(nodes)] = nodes
            return {"nodes": s["nodes"], "count": len(nodes), "tris": b.packed_tris(), "bounds": list(b.bounds())}
    if kind == "rebuild":
        with pkg.BVH.build_device(s["v"], int(s["i"].shape[0]), s["i"]) as b:
            b.trace_pinhole_closest(case["width"], case["height"], s["cam"], s["t"], s["id"], s["u"], s["v2"])
            return {"t": s["t"], "id": s["id"], "u": s["u"], "v": s["v2"], "nodes": b.num_bvh4_nodes, "depth": b.depth}
    if kind == "tlas":
        nodes, order = pkg.build_tlas_fast(s["aabbs"])
        return {"nodes": nodes, "order": order}
    if kind == "scene_rays":
        s["scene"].trace_closest(s["rays"], s["t"], s["inst"], s["prim"], s["u"], s["v"])
        s["scene"].trace_any(s["shadow"], s["occ"])
        return {k: s[k] for k in ("t", "inst", "prim", "u", "v", "occ")}
    if kind == "path":
        s["scene"].path_trace(s["cam"], s["params"], s["rgb"], s["alb"], s["nrm"], s["dep"], flags=pkg.FLAG_GRAPH)
        return {k: s[k] for k in ("rgb", "alb", "nrm", "dep")}
    if kind == "batch_trace":
        s["batch"].trace_closest(s["n"], s["off"], s["rays"], s["t"], s["id"], s["u"], s["v"], flags=pkg.FLAG_GRAPH)
        return {k: s[k] for k in ("t", "id", "u", "v")}
    if kind == "batch_build":
        b = pkg.Batch(s["tris"])
        b.trace_any(s["n"], s["off"], s["rays"], s["occ"])
        roots = b.roots()
        b.destroy()
        return {"occ": s["occ"], "roots": roots}
    if kind == "denoise":
        s["dn"].denoise(case["width"], case["height"], *s["planes"], s["out"])
        return s["out"]
    S = case["size"]
    s["dn"].train_step(case["batch"], S, S, s["x"], s["y"], 1e-8, want_loss=False)
    return {"grads": s["dn"].params(1)}


# ------------------------------------------------------------------- work ----
# (cin, cout, taps, level) of the denoiser's layers
LAYERS = ((10, 32, 9, 0), (32, 32, 9, 0), (32, 64, 9, 1), (64, 64, 9, 1), (64, 128, 9, 2), (128, 128, 9, 2),
          (128, 256, 9, 3), (256, 256, 9, 3), (384, 128, 9, 2), (128, 128, 9, 2), (192, 64, 9, 1), (64, 64, 9, 1),
          (96, 32, 9, 0), (32, 32, 9, 0), (32, 3, 1, 0))
# the first layer's rows are stored 16 channels wide
PARAMS = sum((16 if j == 0 else ci) * co * t + co for j, (ci, co, t, _) in enumerate(LAYERS))


def _tree_bytes(tris):
    """BVH4 nodes (64 bytes, about one per 8 triangles) and 36-byte triangles."""
    return 44 * tris


def _mesh_tris(case):
    return case["tris"] if "tris" in case else 2 * case["res"] ** 2 + 5120 * case["spheres"]


def _mean_log(lo, hi):
    return (hi - lo) / math.log(hi / lo)


def work(case):
    """Tracing: rays in, hits out, and the tree once (or what the rays visit
    of it, about 15 nodes and 6 triangles each, where that is less). Building:
    triangles in, nodes and leaf-order triangles out."""
    kind = case["kind"]
    visit = lambda tris, rays: min(_tree_bytes(tris), rays * (15 * 64 + 6 * 36))     # noqa: E731
    if kind == "rays":
        return dict(bytes=case["rays"] * (32 + (1 if case["any_hit"] else 16)) + visit(case["tris"], case["rays"]), flops=0)
    if kind == "frame":
        n = case["width"] * case["height"]
        return dict(bytes=n * 16 + int(0.5 * n) * (64 + 4 + 64 + 17) + visit(_mesh_tris(case), 2 * n), flops=0)
    if kind == "build":
        return dict(bytes=case["tris"] * (36 + 8 + 48), flops=0)
    if kind == "rebuild":
        t, n = _mesh_tris(case), case["width"] * case["height"]
        return dict(bytes=t * (36 + 8 + 48) + n * 16 + visit(t, n), flops=0)
    if kind == "tlas":
        return dict(bytes=case["boxes"] * (24 + 64 + 4), flops=0)
    if kind == "scene_rays":
        return dict(bytes=case["rays"] * (32 + 20 + 32 + 1) + visit(759622, 2 * case["rays"]), flops=0)
    if kind == "path":
        n = case["width"] * case["height"]
        return dict(bytes=n * 40 + case["spp"] * visit(759622, 2 * n), flops=0)
    if kind in ("batch_trace", "batch_build"):
        tris = case["scenes"] * _mean_log(1000, case["tris_max"])
        if kind == "batch_trace":
            rays = case["scenes"] * (_mean_log(65536, case["rays_max"]) if case["rays_max"] > 65536 else 65536)
            return dict(bytes=rays * 48 + visit(tris, rays), flops=0)
        rays = case["scenes"] * _mean_log(4096, case["rays_max"])
        return dict(bytes=tris * (36 + 8 + 48) + rays * 33 + visit(tris, rays), flops=0)
    W, H = (case["width"], case["height"]) if kind == "denoise" else (case["size"], case["size"])
    macs = sum(ci * co * t * (W >> lv) * (H >> lv) for ci, co, t, lv in LAYERS)
    if kind == "denoise":
        return dict(bytes=W * H * 52 + 2 * PARAMS, flops=2 * macs)
    # forward, input gradients (all but the first layer) and weight gradients
    first = 10 * 32 * 9 * W * H
    return dict(bytes=case["batch"] * W * H * (32 + 12) + PARAMS * 4 * 7, flops=2 * case["batch"] * (3 * macs - first))


# ------------------------------------------------------------------ exact ----
def _brute_closest(tri, o, d):
    """Closest hit t, u, v (miss: 1e30, 0, 0) in float64, every ray against
    every triangle (Moller-Trumbore). tri (m, 9), o and d (3, n) float64."""
    m, n = tri.shape[0], o.shape[1]
    v0, e1, e2 = tri[:, 0:3], tri[:, 3:6] - tri[:, 0:3], tri[:, 6:9] - tri[:, 0:3]
    c = [x.unbind(1) for x in (v0, e1, e2)]
    v0, e1, e2 = [[a[:, None] for a in x] for x in c]
    out = torch.empty(3, n, device=o.device, dtype=torch.float64)
    step = max(1, (1 << 26) // m)
    for b in range(0, n, step):
        O, D = o[:, b:b + step], d[:, b:b + step]
        px, py, pz = (D[1] * e2[2] - D[2] * e2[1], D[2] * e2[0] - D[0] * e2[2], D[0] * e2[1] - D[1] * e2[0])
        inv = 1.0 / (e1[0] * px + e1[1] * py + e1[2] * pz)
        tx, ty, tz = (O[k] - v0[k] for k in range(3))
        u = (tx * px + ty * py + tz * pz) * inv
        qx, qy, qz = ty * e1[2] - tz * e1[1], tz * e1[0] - tx * e1[2], tx * e1[1] - ty * e1[0]
        v = (D[0] * qx + D[1] * qy + D[2] * qz) * inv
        t = (e2[0] * qx + e2[1] * qy + e2[2] * qz) * inv
        t = torch.where((u >= 0) & (v >= 0) & (u + v <= 1) & (t >= 0), t, torch.full_like(t, MISS_T))
        best, at = t.min(0)
        hit = best < MISS_T
        out[0, b:b + step] = best
        out[1, b:b + step] = torch.where(hit, u.gather(0, at[None])[0], torch.zeros_like(best))
        out[2, b:b + step] = torch.where(hit, v.gather(0, at[None])[0], torch.zeros_like(best))
    return out


def _weights64():
    p = torch.from_numpy(denoise_train.load_weights()).to(_dev()).double()
    out, off = [], 0
    for j, (ci, co, taps, _) in enumerate(LAYERS):
        ci = 16 if j == 0 else ci
        w = p[off:off + co * taps * ci].view(co, taps, ci).clone()
        b = p[off + co * taps * ci:off + co * taps * ci + co].clone()
        off += co * taps * ci + co
        out.append((w.requires_grad_(), b.requires_grad_()))
    return out


def _conv64(x, w, b):
    """3x3 (zero padding) or 1x1 convolution, x (B, H, W, C) float64."""
    co, taps, _ = w.shape
    B, H, W, _ = x.shape
    if taps == 1:
        return x @ w[:, 0].t() + b
    p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    y = b.expand(B, H, W, co)
    for t in range(9):
        y = y + p[:, t // 3:t // 3 + H, t % 3:t % 3 + W] @ w[:, t].t()
    return y


def _unet64(x, L):
    def two(x, j):
        return torch.relu(_conv64(torch.relu(_conv64(x, *L[j])), *L[j + 1]))

    def pool(x):
        B, H, W, C = x.shape
        return x.view(B, H // 2, 2, W // 2, 2, C).amax(dim=(2, 4))

    def up(x):
        return x.repeat_interleave(2, 1).repeat_interleave(2, 2)

    e1 = two(x, 0)
    e2 = two(pool(e1), 2)
    e3 = two(pool(e2), 4)
    y = two(pool(e3), 6)
    for j, e in ((8, e3), (10, e2), (12, e1)):
        y = two(torch.cat([up(y), e], -1), j)
    return _conv64(y, *L[14])


def exact(case, seed):
    kind = case["kind"]
    if kind == "rays" and not case["any_hit"] and case["tris"] * case["rays"] <= 1 << 33:
        tri = _soup(case["tris"], seed).double()
        o, d = scenes.batch_rays_device(case["rays"], seed + 1, _dev())
        t, u, v = _brute_closest(tri, o.double(), d.double())
        return {"t": t, "id": None, "u": u, "v": v}
    if kind == "denoise":
        W, H = case["width"], case["height"]
        rgb, alb, nrm, dep, _ = _planes(W, H, seed)
        with torch.no_grad():
            logs = torch.log1p(rgb.double())
            ch = torch.cat([logs, alb.double(), nrm.double(), torch.log1p(dep.double()) * 0.25]).view(10, H, W)
            x = torch.zeros(1, H, W, 16, device=_dev(), dtype=torch.float64)
            x[0, :, :, :10] = ch.permute(1, 2, 0)
            y = _unet64(x, _weights64())
            out = torch.expm1(y[0].permute(2, 0, 1) + logs.view(3, H, W)).clamp_min(0)
        return out.reshape(-1)
    if kind == "train":
        X, Y = _train_data(case, seed)
        x, L = X.double(), _weights64()
        loss = (_unet64(x, L) + x[..., :3] - Y.double()).abs().mean()
        loss.backward()
        return {"grads": torch.cat([g.grad.reshape(-1) for wb in L for g in wb])}
    return None
