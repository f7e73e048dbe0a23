"""Timed workloads of the framework, each through the entry points a program calls.

A case is a dict of plain values.  ``listed()`` names the fixed ones, ``draw(rng)`` makes one more
of the same ranges.  ``prepare`` builds the scene, the renderer and the inputs from the seed (the
work a program does once), ``run`` is one pass, ``work`` the bytes and operations a pass cannot do
without, and ``exact`` the same outputs evaluated in 64 bits by plain torch where the scene is
small enough to test every ray against every triangle.

Kinds:
  cast     DeviceScene.cast over a ray batch resident in device memory
  frame    DumbRenderer.render into a BlockBasedFrameBuffer, benchmark plugins (Lambert, mirror,
           metal, quad lights) or the reference plugins (DumbBasedShader and its siblings,
           directional, spherical and spot lights)
  adjoint  DumbRenderer.backward of a frame gradient
  train    one optimisation step: autograd render, a squared loss, gradients
  batch    RenderBatch.run over many uneven requests
  bytes    images.frame_to_rgba8 of a finished frame
"""
import math

import numpy as np
import torch

import dumbray_amd as D
from dumbray_amd import images, plugins
from dumbray_amd import scenes as S
from dumbray_amd.autograd import render as autograd_render

FLT_MAX = float(np.finfo(np.float32).max)
EPS = 0.000005                      # the framework's vector epsilon
INSIDE_TOL = 32 * EPS               # tolerance of its point-in-triangle test
PAIRS_EXACT = 4e10                  # ray-triangle pairs that exact() tests in well under 20 s


def listed():
    return [
        # a click in a viewer: the rays of an 8x8 pixel patch; latency is all that counts
        dict(name="pick_64", kind="cast", scene="spheres", size=8, rays=64, source="patch", clip=True, points=True),
        # bounce rays leaving a mesh's surface, the triangle they leave excluded; an odd count
        dict(name="cast_bounce_99991", kind="cast", scene="icospheres", size=5, rays=99991, source="surface",
             clip=False, points=True),
        # the primary rays of a 1080p view over a 2M-triangle terrain
        dict(name="cast_primary_1080p", kind="cast", scene="terrain", size=1024, rays=1920 * 1080, source="camera",
             clip=True, points=False),
        # the benchmark's headline batch: 4M rays of no order through the same terrain
        dict(name="cast_incoherent_4M", kind="cast", scene="terrain", size=1024, rays=1 << 22, source="volume",
             clip=False, points=False),
        # interactive preview: one more sample per pixel blended into an odd-sized frame
        dict(name="preview_517x389", kind="frame", plugins="benchmark", scene="icospheres", size=6, width=517,
             height=389, fsaa=1, depth=4, iteration=3),
        # the small benchmark frame
        dict(name="frame_256_4spp", kind="frame", plugins="benchmark", scene="spheres", size=8, width=256, height=256,
             fsaa=2, depth=4, iteration=1),
        # the large benchmark frame: a final-quality 1080p picture with Russian roulette
        dict(name="frame_1080p_16spp", kind="frame", plugins="benchmark", scene="icospheres", size=7, width=1920,
             height=1080, fsaa=4, depth=8, iteration=1),
        # a scene with the reference's own shaders and lights at 1080p
        dict(name="plugins_1080p", kind="frame", plugins="reference", scene="icospheres", size=4, width=1920,
             height=1080, fsaa=1, depth=2, iteration=1),
        # gradients of a rendered image to 64 materials and 4 lights
        dict(name="adjoint_512_16spp", kind="adjoint", scene="spheres", size=64, lights=4, width=512, height=512,
             fsaa=4, depth=4),
        # one step of an inverse-rendering loop at low resolution
        dict(name="train_128_4spp", kind="train", scene="spheres", size=8, lights=1, width=128, height=128, fsaa=2,
             depth=3),
        # a service's queue of uneven requests over several scenes
        dict(name="batch_24", kind="batch", requests=24, scenes=3, largest=512),
        # the finished frame as picture bytes
        dict(name="rgba8_1080p", kind="bytes", width=1920, height=1080),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["cast", "cast", "cast", "frame", "frame", "frame", "adjoint", "train", "batch", "bytes"])
    if kind == "cast":
        scene = rng.choice(["spheres", "icospheres", "terrain"])
        size = {"spheres": lambda: _log_int(rng, 4, 128), "icospheres": lambda: rng.randint(3, 7),
                "terrain": lambda: _log_int(rng, 48, 1024)}[scene]()
        return dict(kind=kind, scene=scene, size=size, rays=_log_int(rng, 64, 1 << 22),
                    source=rng.choice(["patch", "surface", "camera", "volume"]), clip=rng.random() < 0.5,
                    points=rng.random() < 0.5)
    if kind == "frame":
        which = rng.choice(["benchmark", "benchmark", "reference"])
        scene = rng.choice(["spheres", "icospheres"])
        fsaa = rng.choice([1, 1, 2, 3, 4])
        # at most half the samples of a 1080p frame at 16 per pixel, a quarter of that with the reference plugins
        most = 16_000_000 if which == "benchmark" else 4_000_000
        pixels = _log_int(rng, 64 * 64, min(1920 * 1080, most // (fsaa * fsaa)))
        width = max(24, int(math.sqrt(pixels * rng.uniform(0.6, 2.0))))
        return dict(kind=kind, plugins=which, scene=scene,
                    size=_log_int(rng, 4, 128) if scene == "spheres" else rng.randint(3, 7),
                    width=width, height=max(24, pixels // width), fsaa=fsaa,
                    depth=rng.randint(1, 8) if which == "benchmark" else rng.randint(1, 3),
                    iteration=rng.choice([1, 1, 2, 7]))
    if kind in ("adjoint", "train"):
        fsaa = rng.choice([1, 2, 3, 4])
        pixels = _log_int(rng, 48 * 48, (4_000_000 if kind == "adjoint" else 600_000) // (fsaa * fsaa))
        width = max(24, int(math.sqrt(pixels * rng.uniform(0.6, 2.0))))
        return dict(kind=kind, scene="spheres", size=_log_int(rng, 4, 128), lights=rng.randint(1, 4), width=width,
                    height=max(24, pixels // width), fsaa=fsaa, depth=rng.randint(1, 6))
    if kind == "batch":
        return dict(kind=kind, requests=_log_int(rng, 4, 48), scenes=rng.randint(1, 4), largest=rng.choice([128, 256, 512]))
    return dict(kind=kind, width=_log_int(rng, 64, 3840), height=_log_int(rng, 48, 2160))


# ---------------------------------------------------------------- scenes and inputs
def _scene(case, seed):
    """Triangles, materials, lights and camera of the case's scene."""
    if case["scene"] == "terrain":
        cells = case["size"]
        tris = S.heightfield(cells, seed=seed)
        top, bottom = float(tris[:, 1::3].max()), float(tris[:, 1::3].min())
        cam = S.Camera.look_at((0.5 * cells, top + 0.35 * cells, -0.25 * cells), (0.5 * cells, bottom, 0.55 * cells))
        return S.Scene(tris, np.zeros(len(tris), np.int32), [dict(kind="lambert", albedo=(0.5, 0.5, 0.5))], [], cam)
    if case["scene"] == "icospheres":
        return S.icosphere_scene(case["size"], seed=seed)
    return S.spheres_scene(case["size"], seed=seed, n_lights=case.get("lights", 1), ground_material="lights" not in case)


def _knobs(case):
    """Octree settings: the reference's defaults for the icospheres, larger leaves elsewhere."""
    return (8, 24) if case["scene"] == "icospheres" else (16, 12)


def _upload(case, sc):
    tree = D.Octree(*_knobs(case))
    tree.push(sc.tris)
    return tree.build().upload()


def _rays(case, sc, seed):
    """(rays (n, 6), excluded triangle per ray or None) as host arrays."""
    n, rng = case["rays"], np.random.default_rng(seed + 1)
    if case["source"] == "volume":
        return S.incoherent_rays(sc.tris, n, seed=seed + 1), None
    if case["source"] == "surface":
        # cosine-free hemisphere directions off random points of random triangles, on the side
        # that faces rays from outside (-n)
        tri = rng.integers(0, len(sc.tris), n)
        a, b, c = (sc.tris[tri, 3 * k:3 * k + 3].astype(np.float64) for k in range(3))
        u, v = np.sqrt(rng.random((n, 1))), rng.random((n, 1))
        o = a * (1 - u) + b * (u * (1 - v)) + c * (u * v)
        d = rng.normal(size=(n, 3))
        d /= np.linalg.norm(d, axis=1, keepdims=True)
        d *= np.where(np.einsum("ij,ij->i", d, np.cross(b - a, c - a)) > 0, -1.0, 1.0)[:, None]
        return np.ascontiguousarray(np.concatenate([o, d], 1).astype(np.float32)), tri.astype(np.int32)
    if case["source"] == "patch":
        # n pixels of a square patch of a 1080p view, about a point of the mesh in front of the camera
        side = int(math.ceil(math.sqrt(n)))
        w, h = max(1920, side), max(1080, side)
        cam = sc.camera.as_array().astype(np.float64)
        at = (sc.tris[rng.integers(0, len(sc.tris), 256)].reshape(-1, 3, 3).mean(1) - cam[:3]) @ cam[3:12].reshape(3, 3).T
        px = at[at[:, 2] > 0][0] * cam[12] / at[at[:, 2] > 0][0][2]
        x0 = int(np.clip(px[0] * h + w / 2 - side / 2, 0, w - side))
        y0 = int(np.clip(h / 2 - px[1] * h - side / 2, 0, h - side))
        x, y = x0 + np.arange(n) % side, y0 + np.arange(n) // side
    else:
        # the pixels of a whole 16:9 view of n pixels, in rows
        w = max(1, int(round(math.sqrt(n * 16 / 9))))
        h = -(-n // w)
        x, y = np.arange(n) % w, np.arange(n) // w
    cam = sc.camera.as_array().astype(np.float64)
    sx, sy = (x - w / 2 + 0.5) / h, (h / 2 - y - 0.5) / h
    jit = (rng.random((2, n)) - 0.5) / h
    l = np.stack([sx + jit[0], sy + jit[1], np.full(n, cam[12])], 1)
    l /= np.linalg.norm(l, axis=1, keepdims=True)
    d = l @ cam[3:12].reshape(3, 3)
    return np.ascontiguousarray(np.concatenate([np.broadcast_to(cam[:3], (n, 3)), d], 1).astype(np.float32)), None


def _reference_plugins(sc, seed):
    """Materials and lights of the reference's own kinds over the scene's material ids."""
    rng = np.random.default_rng(seed + 2)
    colour = lambda: tuple(float(v) for v in rng.uniform(0.3, 0.9, 3))
    kinds = [lambda: plugins.matte_finish(), lambda: plugins.dumb_based_shader(colour(), 64.0, colour(), 0.2),
             lambda: plugins.simple_stochastic_shader(colour(), 0.6, 0.3, 8.0), lambda: plugins.rough_gold(),
             lambda: plugins.default_shader(colour()), lambda: plugins.fresnel_shader(colour())]
    mats = [kinds[k % len(kinds)]() for k in range(int(sc.mat_id.max()) + 1)]
    lights = [plugins.soft_directional_light((0.8, 0.8, 0.7), (0.4, -1.0, 0.6), 64.0, 0.1),
              plugins.spherical_light((30.0, 28.0, 25.0), (-3.0, 5.0, -3.0), 0.4),
              plugins.spot_light((1.0, 0.9, 0.8), 60.0, (3.0, 6.0, -3.0), (-0.4, -1.0, 0.4), 20.0, 50.0, samples=2)]
    return mats, lights


def _renderer(case, seed, sc, scene):
    mats, lights = (_reference_plugins(sc, seed) if case.get("plugins") == "reference" else (sc.materials, sc.lights))
    return D.DumbRenderer(scene, sc.mat_id, mats, lights, sc.camera, case["width"], case["height"],
                          (case["fsaa"], case["fsaa"]), case["depth"], rr_start=3, rr_survive=0.75, seed=seed)


def _blocks(width, height):
    return -(-width // 8) * -(-height // 16)


def _frame_data(case, seed):
    """A frame's contents before the pass: the picture so far, zeros outside the image."""
    gen = torch.Generator(device="cuda").manual_seed(seed + 3)
    img = torch.rand((case["height"] * case["width"], 4), generator=gen, device="cuda") * 1.2 - 0.05
    out = torch.zeros((_blocks(case["width"], case["height"]) * 128, 4), device="cuda")
    out[_pixel_rows(case["width"], case["height"]).cuda()] = img
    return out


def _pixel_rows(width, height):
    """Row in the block-major frame (8x16-pixel blocks) of every pixel, row by row."""
    y, x = torch.meshgrid(torch.arange(height), torch.arange(width), indexing="ij")
    return (((y // 16) * (-(-width // 8)) + x // 8) * 128 + (y % 16) * 8 + x % 8).reshape(-1)


def _normal(shape, seed):
    return torch.randn(shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda")


def _train_inputs(case, seed, sc):
    gen = torch.Generator().manual_seed(seed + 4)
    albedo = torch.rand((len(sc.materials), 3), generator=gen) * 0.6 + 0.2
    emission = torch.rand((len(sc.lights), 3), generator=gen) * 10.0 + 5.0
    target = torch.rand((_blocks(case["width"], case["height"]) * 128, 3), generator=gen) * 0.02
    return albedo.cuda(), emission.cuda(), target.cuda()


def _requests(case, seed):
    """Scene levels and requests: the mix of sizes follows from the case, the seeds from the seed."""
    rng = np.random.default_rng(1000 * case["requests"] + case["largest"])
    levels = [int(v) for v in rng.permutation([4, 5, 6, 6])[:case["scenes"]]]
    sizes = [v for v in (128, 256, 512) if v <= case["largest"]]
    return levels, [dict(scene=i % len(levels), width=int(rng.choice(sizes)), height=int(rng.choice(sizes)),
                         fsaa=int(rng.choice([1, 2, 4])), depth=int(rng.choice([2, 4, 8])), seed=seed + i)
                    for i in range(case["requests"])]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "bytes":
        frame = D.BlockBasedFrameBuffer(case["width"], case["height"])
        frame.data.copy_(_frame_data(case, seed))
        return dict(kind=kind, frame=frame)
    if kind == "batch":
        levels, reqs = _requests(case, seed)
        scs = [S.icosphere_scene(level, seed=seed + k) for k, level in enumerate(levels)]
        dev = [_upload(dict(scene="icospheres"), sc) for sc in scs]
        frames = [D.BlockBasedFrameBuffer(q["width"], q["height"]) for q in reqs]
        batch = D.RenderBatch([(_renderer(q, q["seed"], scs[q["scene"]], dev[q["scene"]]), f, 1, i + 1)
                               for i, (q, f) in enumerate(zip(reqs, frames))])
        return dict(kind=kind, batch=batch, frames=frames)
    sc = _scene(case, seed)
    scene = _upload(case, sc)
    if kind == "cast":
        rays, exclude = _rays(case, sc, seed)
        return dict(kind=kind, scene=scene, rays=torch.from_numpy(rays).cuda(),
                    args=dict(clip_backfaces=case["clip"], points=case["points"],
                              exclude=None if exclude is None else torch.from_numpy(exclude).cuda()))
    renderer = _renderer(case, seed, sc, scene)
    if kind == "frame":
        frame = D.BlockBasedFrameBuffer(case["width"], case["height"])
        if case["iteration"] > 1:
            frame.data.copy_(_frame_data(case, seed))
        return dict(kind=kind, renderer=renderer, frame=frame, iteration=case["iteration"])
    if kind == "adjoint":
        return dict(kind=kind, renderer=renderer,
                    dl=_normal((_blocks(case["width"], case["height"]) * 128, 4), seed + 6))
    albedo, emission, target = _train_inputs(case, seed, sc)
    return dict(kind=kind, renderer=renderer, albedo=albedo.requires_grad_(True),
                emission=emission.requires_grad_(True), target=target)


def run(state):
    kind = state["kind"]
    if kind == "cast":
        return state["scene"].cast(state["rays"], **state["args"])
    if kind == "frame":
        return state["renderer"].render(state["frame"], state["iteration"]).data
    if kind == "adjoint":
        return state["renderer"].backward(state["dl"])
    if kind == "train":
        img = autograd_render(state["albedo"], state["emission"], state["renderer"])
        loss = ((img[:, :3] - state["target"]) ** 2).sum()
        return (img, *torch.autograd.grad(loss, [state["albedo"], state["emission"]]))
    if kind == "batch":
        state["batch"].run()
        return [f.data for f in state["frames"]]
    return images.frame_to_rgba8(state["frame"])


# ---------------------------------------------------------------- what a pass cannot do without
def _triangles(scene, size):
    return {"terrain": 2 * size * size, "icospheres": 2 + 3 * 20 * 4 ** size, "spheres": 2 + 256 * size}[scene]


def _cast_flops(tris):
    """One descent through a tree of eight children (a box test a level) and one triangle test."""
    return 24 * math.log(max(tris, 8), 8) + 60


def work(case):
    """Lower bounds: the scene's vertices, the inputs and the results once; for pictures one camera
    ray a sample (bounces and light photons depend on what it hits)."""
    kind = case["kind"]
    if kind == "bytes":
        n = case["width"] * case["height"]
        return dict(bytes=20 * n, flops=4 * n)
    if kind == "batch":
        levels, reqs = _requests(case, 0)
        tris = [_triangles("icospheres", level) for level in levels]
        samples = [q["width"] * q["height"] * q["fsaa"] ** 2 for q in reqs]
        return dict(bytes=36 * sum(tris) + sum(16 * q["width"] * q["height"] for q in reqs),
                    flops=sum(n * _cast_flops(tris[q["scene"]]) for n, q in zip(samples, reqs)))
    tris = _triangles(case["scene"], case["size"])
    if kind == "cast":
        per = 24 + 8 + (12 if case["points"] else 0) + (4 if case["source"] == "surface" else 0)
        return dict(bytes=36 * tris + per * case["rays"], flops=_cast_flops(tris) * case["rays"])
    pixels = case["width"] * case["height"]
    casts = pixels * case["fsaa"] ** 2 * (2 if kind == "train" else 1)
    moved = {"frame": 16 if case.get("iteration", 1) == 1 else 32, "adjoint": 16, "train": 16 + 12 + 16}[kind]
    return dict(bytes=36 * tris + moved * pixels, flops=casts * _cast_flops(tris))


# ---------------------------------------------------------------- the same in 64 bits
def exact(case, seed):
    kind = case["kind"]
    if kind == "bytes":
        return _exact_bytes(case, seed)
    if kind == "batch" or case.get("plugins") == "reference":
        return None
    tris = _triangles(case["scene"], case["size"])
    if kind == "cast":
        if tris * case["rays"] > PAIRS_EXACT:
            return None
        sc = _scene(case, seed)
        rays, exclude = _rays(case, sc, seed)
        r = torch.from_numpy(rays).cuda().double()
        ex = None if exclude is None else torch.from_numpy(exclude).cuda().long()
        ids, t = _closest(_prepare_tris(sc.tris), r[:, :3], r[:, 3:], case["clip"], ex)
        hit = (ids >= 0)[:, None]
        out = {"id": None, "t": t}
        if case["points"]:
            out["point"] = torch.where(hit, r[:, :3] + r[:, 3:] * t[:, None], torch.zeros_like(r[:, :3]))
        return out
    paths = case["width"] * case["height"] * case["fsaa"] ** 2
    lights = case.get("lights", 2 if case["scene"] == "icospheres" else 1)
    if paths * (case["depth"] + 1) * (1 + lights) * tris > PAIRS_EXACT:
        return None
    sc = _scene(case, seed)
    if kind == "train":
        albedo, emission, target = _train_inputs(case, seed, sc)
        a, e = albedo.double().requires_grad_(True), emission.double().requires_grad_(True)
        img = _exact_frame(case, seed, sc, a, e)
        loss = ((img[:, :3] - target.double()) ** 2).sum()
        return (img.detach(), *torch.autograd.grad(loss, [a, e]))
    a = torch.tensor([m["albedo"] for m in sc.materials], device="cuda").double().requires_grad_(True)
    e = torch.tensor([l["emission"] for l in sc.lights], device="cuda").double().requires_grad_(True)
    img = _exact_frame(case, seed, sc, a, e)
    if kind == "adjoint":
        dl = _normal((img.shape[0], 4), seed + 6).double()
        return torch.autograd.grad((img[:, :3] * dl[:, :3]).sum(), [a, e])
    img = img.detach()
    if case["iteration"] > 1:
        old, amount = _frame_data(case, seed).double(), 1.0 / case["iteration"]
        rows = _pixel_rows(case["width"], case["height"]).cuda()
        new = old.clone()
        new[rows] = img[rows] * amount + old[rows] * (1 - amount)
        return new
    return img


def _exact_bytes(case, seed):
    """255 * c in [0, 255], the fraction dropped; the product is rounded to 32 bits, as it is stored."""
    data = _frame_data(case, seed)[_pixel_rows(case["width"], case["height"]).cuda()]
    v = (data.double() * 255.0).float().clamp(0.0, 255.0)
    return v.to(torch.uint8).view(case["height"], case["width"], 4)


def _prepare_tris(tris):
    """Vertices and what the triangle test needs of them, without the degenerate triangles."""
    v = torch.from_numpy(tris).cuda().double()
    a, b, c = v[:, :3], v[:, 3:6], v[:, 6:]
    keep = ~((a == b).all(1) | (b == c).all(1) | (c == a).all(1))
    ids = keep.nonzero()[:, 0]
    a, b, c = a[ids], b[ids], c[ids]
    n = torch.linalg.cross(b - a, c - a)
    edges = []
    for p, e, back in ((a, b - a, a - c), (b, c - b, b - a), (c, a - c, c - b)):
        # a point is inside at this corner if e . (x - p) / |x - p| + tol >= e . (-back) / |back|
        edges.append((p, e, -(e * back).sum(1) / back.norm(dim=1)))
    return ids, a, n, edges


def _closest(T, o, d, clip, exclude):
    """(triangle, distance) of the closest accepted hit of every ray, -1 and FLT_MAX for none."""
    ids, a, n, edges = T
    out_id = torch.full((len(o),), -1, dtype=torch.long, device=o.device)
    out_t = torch.full((len(o),), FLT_MAX, dtype=torch.float64, device=o.device)
    inf = torch.tensor(float("inf"), dtype=torch.float64, device=o.device)
    step = max(1, (1 << 25) // max(len(ids), 1))
    for at in range(0, len(o), step):
        oo, dd = o[at:at + step], d[at:at + step]
        dp = (a * n).sum(1)[None] - oo @ n.T
        dn = dd @ n.T
        ok = dp * dn > 0
        if clip:
            ok &= dp >= -EPS
        t = torch.where(ok, dp / torch.where(ok, dn, torch.ones_like(dn)), torch.zeros_like(dn))
        for p, e, thr in edges:
            q2 = (oo * oo).sum(1)[:, None] - 2 * (oo @ p.T) + (p * p).sum(1)[None]
            qd = (oo * dd).sum(1)[:, None] - dd @ p.T
            s = (q2 + 2 * t * qd + t * t * (dd * dd).sum(1)[:, None]).clamp_min(0)
            along = (oo @ e.T - (p * e).sum(1)[None]) + t * (dd @ e.T)
            ok &= (s == 0) | (along / torch.where(s > 0, s, torch.ones_like(s)).sqrt() + INSIDE_TOL >= thr[None])
        if exclude is not None:
            ok &= ids[None] != exclude[at:at + step, None]
        best, k = torch.where(ok, t, inf).min(1)
        got = torch.isfinite(best)
        out_id[at:at + step] = torch.where(got, ids[k], torch.full_like(k, -1))
        out_t[at:at + step] = torch.where(got, best, torch.full_like(best, FLT_MAX))
    return out_id, out_t


def _uniforms(pix, samp, layer, purpose, seed):
    """The framework's four uniforms of (pixel, sample, layer, purpose): Philox4x32-10, 24 bits each."""
    n, m32 = len(pix), np.uint64(0xFFFFFFFF)
    c = [pix.cpu().numpy().astype(np.uint64), samp.cpu().numpy().astype(np.uint64),
         np.full(n, (layer << 8) | purpose, np.uint64), np.zeros(n, np.uint64)]
    k0, k1 = seed & 0xFFFFFFFF, (seed >> 32) & 0xFFFFFFFF
    for _ in range(10):
        p0, p1 = c[0] * np.uint64(0xD2511F53), c[2] * np.uint64(0xCD9E8D57)
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & m32, (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), p0 & m32]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return [torch.from_numpy((v >> np.uint64(8)).astype(np.float64) / 16777216.0).to(pix.device) for v in c]


def _unit(v):
    return v / v.norm(dim=1, keepdim=True)


def _about(n, u0, u1):
    """Cosine-weighted direction about unit n (the branch-free basis of Duff et al., JCGT 2017)."""
    sign = torch.where(n[:, 2] < 0, -torch.ones_like(u0), torch.ones_like(u0))
    a = -1.0 / (sign + n[:, 2])
    b = n[:, 0] * n[:, 1] * a
    b1 = torch.stack([1.0 + sign * n[:, 0] ** 2 * a, sign * b, -sign * n[:, 0]], 1)
    b2 = torch.stack([b, sign + n[:, 1] ** 2 * a, -n[:, 1]], 1)
    r, ang = u0.sqrt(), 2 * math.pi * u1
    return b1 * (r * ang.cos())[:, None] + b2 * (r * ang.sin())[:, None] + n * (1 - u0).sqrt()[:, None]


def _exact_frame(case, seed, sc, albedo, emission):
    """The path estimator of the benchmark plugins with the framework's random numbers, in 64 bits,
    as a block-major frame; differentiable in albedo and emission."""
    dev, f64 = albedo.device, torch.float64
    W, H, f, depth = case["width"], case["height"], case["fsaa"], case["depth"]
    spp = f * f
    samp0 = (max(case.get("iteration", 1), 1) - 1) * spp
    T = _prepare_tris(sc.tris)
    v = torch.from_numpy(sc.tris).to(dev).double()
    normals = torch.linalg.cross(v[:, 3:6] - v[:, :3], v[:, 6:] - v[:, :3])
    mat = torch.from_numpy(sc.mat_id).to(dev).long()
    kind = torch.tensor([{"lambert": 0, "mirror": 1, "metal": 2}[m["kind"]] for m in sc.materials], device=dev)
    cam = torch.from_numpy(sc.camera.as_array()).to(dev).double()
    quads = [[torch.tensor(l[k], dtype=torch.float32, device=dev).double() for k in ("corner", "edge_u", "edge_v")]
             for l in sc.lights]

    pix = torch.arange(W * H, device=dev).repeat_interleave(spp)
    s = torch.arange(spp, device=dev).repeat(W * H)
    samp = s + samp0
    u = _uniforms(pix, samp, 0, 0, seed)
    x, y, ps = (pix % W).double(), (pix // W).double(), 1.0 / H
    pd = ps / f
    lx = (x - W / 2) * ps + ((s // f).double() + 0.5) * pd + (u[0] - 0.5) * pd
    ly = (H / 2 - y) * ps + ((s % f).double() + 0.5) * pd + (u[1] - 0.5) * pd
    d = lx[:, None] * cam[3:6] + ly[:, None] * cam[6:9] + cam[12] * cam[9:12]
    o = cam[:3].expand_as(d)
    row = torch.arange(len(pix), device=dev)          # the path each active entry belongs to
    beta = torch.ones((len(pix), 3), dtype=f64, device=dev)
    excl = torch.full((len(pix),), -1, dtype=torch.long, device=dev)
    L = torch.zeros((len(pix), 3), dtype=f64, device=dev)
    for layer in range(depth + 1):
        h, t = _closest(T, o, d, True, excl)
        on = (h >= 0).nonzero()[:, 0]
        if not len(on):
            break
        h, row, beta = h[on], row[on], beta[on]
        p = o[on] + d[on] * t[on, None]
        du, nu = _unit(d[on]), _unit(normals[h])
        nu = torch.where((nu * du).sum(1, keepdim=True) > 0, -nu, nu)
        m = mat[h]
        lam = kind[m] == 0
        for l, (corner, eu, ev) in enumerate(quads):
            w = lam.nonzero()[:, 0]
            u = _uniforms(pix[row[w]], samp[row[w]], layer, 16 + l, seed)
            q = corner + eu * u[0][:, None] + ev * u[1][:, None]
            delta = p[w] - q
            d2 = (delta * delta).sum(1)
            wi = delta / d2.sqrt()[:, None]
            nl = torch.linalg.cross(eu, ev)
            area = nl.norm()
            cos_l, cos_i = (wi * (nl / area)).sum(1), -(wi * nu[w]).sum(1)
            g = ((cos_l > 0) & (cos_i > 0)).nonzero()[:, 0]
            hh, tt = _closest(T, q[g], wi[g], True, None)
            e = q[g] + wi[g] * tt[:, None] - p[w[g]]
            lit = (hh >= 0) & ((hh == h[w[g]]) | ((e * e).sum(1) <= 8 * EPS))
            g = g[lit]
            at = w[g]
            k = (cos_i[g] / math.pi * cos_l[g] * area / d2[g])[:, None]
            L = L.index_add(0, row[at], beta[at] * albedo[m[at]] * emission[l] * k)
        if layer >= depth:
            break
        u = _uniforms(pix[row], samp[row], layer, 1, seed)
        sd = torch.where(lam[:, None], _about(nu, u[0], u[1]), du - nu * (2 * (du * nu).sum(1, keepdim=True)))
        f5 = torch.where(kind[m] == 2, (1 - (nu * sd).sum(1)) ** 5, torch.zeros_like(u[0]))[:, None]
        A = albedo[m] + (1 - albedo[m]) * f5
        weight, stay = 1.0, torch.ones(len(row), dtype=torch.bool, device=dev)
        if layer >= 3:                                # Russian roulette, as _renderer sets it
            weight, stay = 1.0 / 0.75, u[2] < 0.75
        keep = stay.nonzero()[:, 0]
        beta, row, o, d, excl = (beta * A * weight)[keep], row[keep], p[keep], sd[keep], h[keep]
    img = L.view(W * H, spp, 3).sum(1) / spp
    out = torch.zeros((_blocks(W, H) * 128, 4), dtype=f64, device=dev)
    return out.index_copy(0, _pixel_rows(W, H).to(dev), torch.cat([img, torch.ones_like(img[:, :1])], 1))
