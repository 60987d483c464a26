"""Workloads whose time matters to a user of the ray tracer, and their checks.

Three kinds of program use it: one that brings its own ray streams and
shades the hits itself (`gpu.trace_rays`, `gpu.trace_world`,
`gpu.intersections`), one that renders images (`gpu.render`), and one that
fits scene parameters to an image (`diff.render_image` with its backward
pass).  The scenes are the ones `psychopath_cpp_amd.configs` defines, with
their sizes, options (dicing rate, motion, depth of field, instancing, many
lights) and path lengths; everything is float32, the only type there is.
All of them run with the library's defaults, as a program that calls it
without tuning gets them.
"""
import math

import numpy as np
import torch

from psychopath_cpp_amd import abi, configs, diff, gpu, scene

EXTENT = 10.0                # side of the terrain
EYE, TARGET, FOV = (0.0, -1.5, 11.5), (0.0, 0.3, 0.0), math.radians(36.0)  # configs.heightfield_scene's camera
LIGHT_POS, LIGHT_SIZE = (0.0, -3.0, 13.5), 2.0
FAR = 1.00000024             # slack of a box's far distance
MIN_UPOLY = 1e-5             # smallest micropolygon


def listed():
    return [
        # the smallest call: a 48x48 tile of world rays, e.g. a preview or a pick under the cursor; launches count
        {"name": "trace-tile", "kind": "world", "scene": "terrain", "grid": 16, "dice_rate": 0.25, "width": 48,
         "height": 48, "spp": 1, "bounce": False, "shade": False},
        # the headline stream: 2^21 camera and 2^21 bounce rays in their 56-byte form through the 64x64 heightfield
        {"name": "trace-stream", "kind": "rays", "scene": "terrain", "grid": 64, "dice_rate": 1.0, "width": 1024,
         "height": 1024, "spp": 2, "bounce": True},
        # a program with its own shading: odd-sized image of Catmull-Clark surfaces, hits and then their full records
        {"name": "shade-subdivision", "kind": "world", "scene": "subdivision", "grid": 64, "dice_rate": 0.25,
         "width": 641, "height": 479, "spp": 1, "bounce": False, "shade": True},
        # camera rays of one ordinary frame through instanced, moving bicubic patches with depth of field
        {"name": "trace-motion", "kind": "world", "scene": "motion", "grid": 32, "dice_rate": 1.0, "width": 960,
         "height": 540, "spp": 1, "bounce": False, "shade": False},
        # any-hit shadow rays between points of the sphere scene (a program that does its own direct light)
        {"name": "trace-shadow", "kind": "shadow", "scene": "spheres", "spheres": 64, "rays": 1000003},
        # a preview render: the smallest image, every step of the wavefront nearly empty
        {"name": "render-preview", "kind": "render", "scene": "spheres", "spheres": 64, "width": 96, "height": 64,
         "spp": 1, "path_length": 4},
        # an odd-sized crop of the heightfield at the reference's dicing rate, one sample
        {"name": "render-crop", "kind": "render", "scene": "terrain", "grid": 64, "dice_rate": 0.25, "width": 331,
         "height": 173, "spp": 3, "path_length": 4},
        # the four configurations: spheres at its own size, the others at the sizes their figures are quoted on
        {"name": "render-spheres", "kind": "render", "scene": "spheres", "spheres": 64, "width": 256, "height": 256,
         "spp": 16, "path_length": 4},
        {"name": "render-terrain", "kind": "render", "scene": "terrain", "grid": 64, "dice_rate": 1.0, "width": 1024,
         "height": 1024, "spp": 16, "path_length": 4},
        {"name": "render-motion", "kind": "render", "scene": "motion", "grid": 64, "dice_rate": 1.0, "width": 960,
         "height": 540, "spp": 8, "path_length": 6},
        {"name": "render-lights", "kind": "render", "scene": "lights", "lights": 10000, "width": 1024,
         "height": 1024, "spp": 4, "path_length": 4},
        # one step of a fit: image, loss and the gradients of 257 albedos and 1000 emissions
        {"name": "fit-lights", "kind": "fit", "scene": "fit", "spheres": 256, "lights": 1000, "width": 512,
         "height": 512, "spp": 16, "path_length": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges; none has more samples than the largest listed one of its kind."""
    kind = rng.choice(["world", "rays", "shadow", "render", "render", "render", "fit"])
    width = _log(rng, 48, 1024)
    height = max(32, int(width * rng.uniform(0.5, 1.0)))
    spp = _log(rng, 1, 16)
    if kind == "shadow":
        return {"kind": kind, "scene": "spheres", "spheres": _log(rng, 16, 256), "rays": _log(rng, 2000, 2000000)}
    if kind == "fit":
        width, height = min(width, 512), min(height, 512)
        return {"kind": kind, "scene": "fit", "spheres": _log(rng, 16, 256), "lights": _log(rng, 10, 1000),
                "width": width, "height": height, "spp": spp, "path_length": rng.randint(2, 4)}
    dice = rng.choice([0.25, 1.0])
    if kind in ("world", "rays"):
        name = "terrain" if kind == "rays" else rng.choice(["terrain", "subdivision", "motion"])
        c = {"kind": kind, "scene": name, "grid": _log(rng, 12, 64), "dice_rate": dice, "width": width,
             "height": height, "spp": rng.randint(1, 2), "bounce": name == "terrain" and rng.random() < 0.5}
        if name == "motion":
            c.update(grid=_log(rng, 12, 32), width=min(width, 960), height=min(height, 540), spp=1)
        if kind == "world":
            c["shade"] = rng.random() < 0.5
        return c
    name = rng.choice(["terrain", "spheres", "motion", "lights"])
    c = {"kind": kind, "scene": name, "width": width, "height": height, "spp": spp, "path_length": rng.randint(2, 4)}
    if name == "terrain":
        c.update(grid=_log(rng, 12, 64), dice_rate=dice)
    elif name == "spheres":
        c.update(spheres=_log(rng, 16, 256))
    elif name == "lights":
        c.update(lights=_log(rng, 100, 10000), spp=min(spp, 4))
    else:
        c.update(grid=_log(rng, 12, 64), dice_rate=1.0, width=min(width, 960), height=min(height, 540),
                 spp=min(spp, 8), path_length=rng.randint(2, 6))
    return c


# ---- scenes ------------------------------------------------------------------
def _terrain(grid, seed):
    """(grid + 1)^2 float32 vertices of a sum of eight sines, as configs.heightfield draws its own."""
    rng = np.random.default_rng(seed)
    xs = np.linspace(-EXTENT / 2, EXTENT / 2, grid + 1)
    X, Y = np.meshgrid(xs, xs, indexing="xy")
    Z = np.zeros_like(X)
    for _ in range(8):
        a, f = rng.uniform(0.05, 0.3), rng.uniform(1.0, 8.0)
        th, ph = rng.uniform(0.0, 2 * math.pi, 2)
        Z += a * np.sin(f * (X * math.cos(th) + Y * math.sin(th)) + ph)
    return np.stack([X, Y, Z], -1).astype(np.float32)


def _terrain_patches(grid, seed):
    """(grid^2, 4, 3): the corners v1 v2 v3 v4 of every quad."""
    V = _terrain(grid, seed)
    return np.stack([V[:-1, :-1], V[:-1, 1:], V[1:, :-1], V[1:, 1:]], 2).reshape(-1, 4, 3)


def _build(case, seed):
    """The case's scene; `seed` places and shapes everything in it."""
    name = case["scene"]
    if name == "terrain":
        root = scene.Assembly()
        sc = scene.Scene(scene.Camera([scene.look_at(EYE, TARGET)], [FOV]), root, dice_rate=case["dice_rate"])
        sc.add_surface_shader("ground", abi.PSY_SHADER_LAMBERT, (0.5, 0.5, 0.5))
        for i, p in enumerate(_terrain_patches(case["grid"], seed)):
            root.add_object(f"p{i}", scene.Bilinear(p))
            root.create_object_instance(f"p{i}", [], "ground")
        root.add_object("light", scene.RectangleLight(LIGHT_SIZE, LIGHT_SIZE, (20.0, 20.0, 20.0)))
        root.create_object_instance("light", [scene.translate(*LIGHT_POS)], None)
        return sc
    if name == "subdivision":
        return configs.subdivision_scene(seed=seed, grid=case["grid"], dice_rate=case["dice_rate"])
    if name == "motion":
        return configs.bicubic_sphere_scene(seed=seed, grid=case["grid"], dice_rate=case["dice_rate"])
    if name == "spheres":
        return configs.sphere_scene(seed=seed, n_spheres=case["spheres"])
    if name == "lights":
        return configs.many_light_scene(seed=seed, n_lights=case["lights"])
    return configs.adjoint_scene(seed=seed, n_spheres=case["spheres"], n_lights=case["lights"])


# ---- ray streams of a program with its own camera (float32, plain torch) -------
def _gen(seed, dev):
    return torch.Generator(device=dev).manual_seed(int(seed))


def _unit(v):
    return v / v.norm(dim=0, keepdim=True)


def _world(o, d, odx, ody, ddx, ddy, g):
    """(20, n) planes: origin, direction, four differentials, time, type."""
    n = o.shape[1]
    time = torch.rand(1, n, generator=g, device=o.device)
    kind = torch.full((1, n), 1, dtype=torch.int32, device=o.device).view(torch.float32)
    return torch.cat([o, d, odx, ody, ddx, ddy, time, kind]).contiguous()


def _camera_stream(case, seed, dev):
    """Pinhole rays through jittered pixel samples, ordered (y, x, sample)."""
    g = _gen(seed, dev)
    W, H, S = case["width"], case["height"], case["spp"]
    f = np.asarray(TARGET) - np.asarray(EYE)
    f = f / np.linalg.norm(f)
    r = np.cross(f, (0.0, 0.0, 1.0))
    r = r / np.linalg.norm(r)
    axes = torch.tensor(np.stack([r, np.cross(r, f), f]), dtype=torch.float32, device=dev)  # right, up, forward
    px = torch.arange(W, device=dev, dtype=torch.float32)[None, :, None]
    py = torch.arange(H, device=dev, dtype=torch.float32)[:, None, None]
    jit = torch.rand(2, H, W, S, generator=g, device=dev)
    tf, step = math.tan(FOV / 2), 2.0 / W
    x = (((px + jit[0]) / W - 0.5) * 2.0 * tf).reshape(1, -1)
    y = ((0.5 - (py + jit[1]) / H) * 2.0 * (H / W) * tf).reshape(1, -1)
    n = x.shape[1]
    d = _unit(axes[0][:, None] * x + axes[1][:, None] * y + axes[2][:, None])
    o = torch.tensor(EYE, dtype=torch.float32, device=dev)[:, None].expand(3, n)
    z = torch.zeros(3, n, device=dev)
    return _world(o, d, z, z, (axes[0] * (step * tf))[:, None].expand(3, n), (axes[1] * (step * tf))[:, None].expand(3, n),
                  g)


def _bounce_stream(case, seed, dev):
    """Cosine-distributed rays off the terrain, from points in scan order."""
    g = _gen(seed + 1, dev)
    W, H, S, grid = case["width"], case["height"], case["spp"], case["grid"]
    P = torch.tensor(_terrain_patches(grid, seed), device=dev)
    q = torch.rand(2, H, W, S, generator=g, device=dev)
    x = ((torch.arange(W, device=dev, dtype=torch.float32)[None, :, None] + q[0]) / W).reshape(-1) * grid
    y = ((torch.arange(H, device=dev, dtype=torch.float32)[:, None, None] + q[1]) / H).reshape(-1) * grid
    i, j = x.long().clamp(max=grid - 1), y.long().clamp(max=grid - 1)
    u, v = (x - i)[:, None], (y - j)[:, None]
    c = P[j * grid + i]
    du = (c[:, 1] - c[:, 0]) * (1 - v) + (c[:, 3] - c[:, 2]) * v
    dv = (c[:, 2] - c[:, 0]) * (1 - u) + (c[:, 3] - c[:, 1]) * u
    p = (c[:, 0] * (1 - u) + c[:, 1] * u) * (1 - v) + (c[:, 2] * (1 - u) + c[:, 3] * u) * v
    nrm = _unit(torch.cross(du, dv, dim=1).T)
    tx = _unit(du.T)
    ty = torch.cross(nrm, tx, dim=0)
    s = torch.rand(2, p.shape[0], generator=g, device=dev)
    rad, ang = s[0].sqrt(), s[1] * (2 * math.pi)
    d = _unit(tx * (rad * ang.cos()) + ty * (rad * ang.sin()) + nrm * (1 - s[0]).clamp(min=1e-6).sqrt())
    a = _unit(torch.cross(d, nrm + 0.5 * tx, dim=0))
    b = torch.cross(d, a, dim=0)
    foot = 0.01 * 1024.0 / W
    return _world(p.T + nrm * 0.02, d, tx * foot, ty * foot, a * 0.15, b * 0.15, g)


def _terrain_rays(case, seed, dev):
    w = _camera_stream(case, seed, dev)
    return torch.cat([w, _bounce_stream(case, seed, dev)], 1).contiguous() if case["bounce"] else w


def _shadow_stream(case, seed, dev):
    """Occlusion rays between two random points of the sphere scene's room (d is the whole segment)."""
    g = _gen(seed, dev)
    n = case["rays"]
    lo = torch.tensor([-10.0, -10.0, 0.2], device=dev)[:, None]
    o = lo + torch.rand(3, n, generator=g, device=dev) * torch.tensor([20.0, 20.0, 4.8], device=dev)[:, None]
    lo = torch.tensor([-8.0, -8.0, 6.0], device=dev)[:, None]
    e = lo + torch.rand(3, n, generator=g, device=dev) * torch.tensor([16.0, 16.0, 3.0], device=dev)[:, None]
    z = torch.zeros(3, n, device=dev)
    w = _world(o, e - o, z + 0.01, z + 0.01, z, z, g)
    w[19] = torch.tensor(abi.PSY_RAY_OCCLUSION, dtype=torch.int32, device=dev).view(torch.float32)
    return w


# ---- the calls -----------------------------------------------------------------
def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    ctx = gpu.Context(dev.index)
    sc = gpu.GpuScene(ctx, _build(case, seed))
    s = {"case": case, "seed": 1 + seed % 100003, "ctx": ctx, "scene": sc}
    kind = case["kind"]
    if kind in ("rays", "world", "shadow"):
        if kind == "shadow":
            w = _shadow_stream(case, seed, dev)
        elif case["scene"] == "terrain":
            w = _terrain_rays(case, seed, dev)
        else:
            w, _ = gpu.camera_rays(ctx, sc, case["width"], case["height"], case["spp"], s["seed"])
        s["rays"] = gpu.world_to_rays(ctx, w) if kind == "rays" else w
        s["hits"] = gpu.HitBuffers(w.shape[1], dev)
    elif kind == "fit":
        g = _gen(seed, dev)
        alb, _ = sc.get_params()
        n_e = sc.param_counts()[1]
        alb = torch.from_numpy(alb).to(dev)
        s["albedo"] = (alb * (0.5 + torch.rand(alb.shape, generator=g, device=dev))).requires_grad_()
        s["emission"] = (0.5 + torch.rand(n_e, generator=g, device=dev)).requires_grad_()
        y = torch.linspace(0.0, 0.6, case["height"], device=dev)[:, None, None]
        s["target"] = y + 0.1 * torch.rand(case["height"], case["width"], 3, generator=g, device=dev)
    return s


def run(state):
    c, ctx, sc = state["case"], state["ctx"], state["scene"]
    if c["kind"] in ("rays", "world", "shadow"):
        if c["kind"] == "rays":
            h = gpu.trace_rays(ctx, sc, state["rays"], hits=state["hits"])
        else:
            h = gpu.trace_world(ctx, sc, state["rays"], hits=state["hits"])
        if c["kind"] == "shadow":
            # which blocker an any-hit ray reports is the tracer's choice; whether there is one is the answer
            return {"blocked": h.inst != -1}
        out = {"t": h.t, "inst": h.inst, "u": h.u, "v": h.v, "aux": h.aux}
        if c.get("shade"):
            out["records"] = gpu.intersections(ctx, sc, state["rays"], h)
        return out
    if c["kind"] == "render":
        film, _, _ = gpu.render(ctx, sc, c["width"], c["height"], c["spp"], state["seed"], c["path_length"])
        return {"film": film}
    film = diff.render_image(ctx, sc, state["albedo"], state["emission"], c["width"], c["height"], c["spp"],
                             state["seed"], c["path_length"])
    loss = ((film - state["target"]) ** 2).sum()
    d_albedo, d_emission = torch.autograd.grad(loss, (state["albedo"], state["emission"]))
    return {"film": film.detach(), "d_albedo": d_albedo, "d_emission": d_emission}


# ---- what a pass cannot do without -----------------------------------------------
def _samples(case):
    return case["width"] * case["height"] * case["spp"]


def _ray_flops(case):
    """One path down a tree of 4-wide nodes over the leaves, then down the split tree to a pixel-sized piece of
    the patch that is hit: 12 operations a box, 4 boxes a node and 2 a split; or the few tens of a sphere."""
    name = case["scene"]
    leaves = {"terrain": case.get("grid", 0) ** 2, "subdivision": case.get("grid", 0) ** 2,
              "motion": 16 * case.get("grid", 0) ** 2, "spheres": case.get("spheres", 0) + 3,
              "lights": case.get("lights", 0) + 67,
              "fit": case.get("spheres", 0) + case.get("lights", 0) + 1}[name]
    nodes = math.ceil(math.log(max(leaves, 4), 4))
    splits = 10 if name in ("terrain", "subdivision", "motion") else 2
    return 12.0 * (4 * nodes + 2 * splits) + 40.0


def work(case):
    kind = case["kind"]
    if kind == "shadow":
        n = case["rays"]
        return {"bytes": n * (80.0 + 1.0), "flops": n * _ray_flops(case)}
    if kind in ("rays", "world"):
        n = _samples(case) * (2 if case["bounce"] else 1)
        # 56-byte or 80-byte rays in, 20-byte hits out, 44 planes of records if wanted
        b = (56.0 if kind == "rays" else 80.0) + 20.0 + (176.0 if case.get("shade") else 0.0)
        return {"bytes": n * b, "flops": n * _ray_flops(case)}
    # Every sample's camera ray, and a shadow and a bounce ray for the half of them that hit something, plus about
    # 1000 operations of sampling and shading a vertex; the film is all that has to leave the chip.
    pixels = case["width"] * case["height"]
    f = _samples(case) * (2.0 * _ray_flops(case) + 1000.0)
    if kind == "fit":
        return {"bytes": pixels * 36.0 + 8.0 * (case["spheres"] + case["lights"]), "flops": 2.0 * f}
    return {"bytes": pixels * 12.0, "flops": f}


def tolerance(case):
    """A hit is the middle of a box's slab interval, the same whatever the order of the walk; of two pieces of a
    patch at exactly the same distance either may be reported, with its own (u, v).  Measured by walking the same
    rays over split trees cached 3 and 7 levels shallower, which changes the order: no distance or instance
    changed, (u, v) by up to 9e-5 (largest single one 0.06), films by up to 6e-5 (largest pixel 0.04), and two
    identical gradient passes, whose sums have no fixed order, by up to 1.1e-6.  Four times that is stated."""
    if case["kind"] == "shadow":
        return {"differ": 1e-5}
    if case["kind"] in ("rays", "world"):
        return {"rel": 4e-4, "max": 0.25, "differ": 1e-5}
    if case["kind"] == "render":
        return {"rel": 2.5e-4, "max": 0.16}
    return {"rel": 1e-5}


# ---- 64 bits -----------------------------------------------------------------------
def _closest_t2(o1, d1, o2, d2):
    dd = d1 - d2
    dd2 = (dd * dd).sum(0)
    t = -((o1 - o2) * dd).sum(0) / dd2
    dist = ((o1 + d1 * t) - (o2 + d2 * t)).norm(dim=0)
    small = dd2 < 1e-5
    return torch.where(small, -1.0, t), torch.where(small, -1.0, dist)


def _footprint(o, d, od, dd):
    """(ow, dw, fw) of one differential: the width is |(ow - fw) + dw t| + fw."""
    t, dist = _closest_t2(o, d, o + od, d + dd)
    ow = od.norm(dim=0)
    ahead = t > 0
    return ow, torch.where(ahead, (dist - ow) / t, dd.norm(dim=0)), torch.where(ahead, dist, 0.0)


def _min_width(w, h0, h1):
    best = None
    for ow, dw, fw in w:
        k = ow - fw
        m = torch.minimum((k + dw * h0).abs(), (k + dw * h1).abs()) + fw
        flip = k / dw
        m = torch.where((h0 < flip) & (h1 > flip), fw, m)
        best = m if best is None else torch.minimum(best, m)
    return best


def _slab(lo, hi, o, inv):
    a, b = (lo - o) * inv, (hi - o) * inv
    h0 = torch.minimum(a, b).amax(1).clamp(min=0.0)
    h1 = torch.maximum(a, b).amin(1) * FAR
    return h0, h1


def _trace64(P, grid, dice_rate, w, t, u, v, aux):
    """Closest hits of world rays w (20, n) on the diced patches P (grid^2, 4, 3), both float64: level by level, the
    pairs of a ray and a piece of a patch whose box it meets, down to the pieces no larger than its footprint."""
    n, dev = w.shape[1], w.device
    o, d = w[0:3], w[3:6]
    inv = (1.0 / d).T
    foot = [_footprint(o, d, w[6:9], w[12:15]), _footprint(o, d, w[9:12], w[15:18])]
    oT = o.T
    # the quadtree of patch boxes, from its root down
    size = 1 << max(0, math.ceil(math.log2(grid)))
    lo = torch.full((size, size, 3), math.inf, dtype=torch.float64, device=dev)
    hi = -lo
    lo[:grid, :grid] = P.amin(1).reshape(grid, grid, 3)
    hi[:grid, :grid] = P.amax(1).reshape(grid, grid, 3)
    levels = [(lo, hi)]
    while levels[-1][0].shape[0] > 1:
        a, b = levels[-1]
        k = a.shape[0] // 2
        levels.append((a.reshape(k, 2, k, 2, 3).amin((1, 3)), b.reshape(k, 2, k, 2, 3).amax((1, 3))))
    ray = torch.arange(n, device=dev)
    cell = torch.zeros(n, dtype=torch.long, device=dev)
    for at in range(len(levels) - 1, -1, -1):
        lo, hi = (x.reshape(-1, 3) for x in levels[at])
        k = levels[at][0].shape[0]
        h0, h1 = _slab(lo[cell], hi[cell], oT[ray], inv[ray])
        keep = (h0 <= h1) & torch.isfinite(lo[cell, 0])
        ray, cell = ray[keep], cell[keep]
        if at:
            y, x = (cell // k) * 2, (cell % k) * 2
            cell = torch.cat([(y + b) * (2 * k) + x + a for b in (0, 1) for a in (0, 1)])
            ray = ray.repeat(4)
    p = P[(cell // size) * grid + cell % size]
    uv = torch.tensor([0.0, 1.0, 0.0, 1.0], dtype=torch.float64, device=dev).repeat(ray.numel(), 1)
    for _ in range(48):
        if not ray.numel():
            break
        lo, hi = p.amin(1), p.amax(1)
        h0, h1 = _slab(lo, hi, oT[ray], inv[ray])
        size_ = (hi - lo).amax(1)
        hit = (h0 <= h1) & (h0 <= t[ray])
        width = (_min_width([tuple(x[ray] for x in f) for f in foot], h0, h1) * dice_rate).clamp(min=MIN_UPOLY)
        leaf = hit & (size_ <= width)
        mid = (h0 + h1) * 0.5
        ok = leaf & (mid > 0)
        r, m = ray[ok], mid[ok]
        t.scatter_reduce_(0, r, m, "amin")
        won = m == t[r]
        r, c = r[won], uv[ok][won]
        u[r], v[r], aux[r] = (c[:, 0] + c[:, 1]) * 0.5, (c[:, 2] + c[:, 3]) * 0.5, size_[ok][won]
        go = hit & ~leaf
        ray, p, uv = ray[go], p[go], uv[go]
        along_u = ((p[:, 0] - p[:, 1]).abs().amax(1) > (p[:, 0] - p[:, 2]).abs().amax(1))[:, None]
        # corners at the halves: v1-v2 and v3-v4 cut along u, v1-v3 and v2-v4 along v
        ma = torch.where(along_u, p[:, 0] + p[:, 1], p[:, 0] + p[:, 2]) * 0.5
        mb = torch.where(along_u, p[:, 2] + p[:, 3], p[:, 1] + p[:, 3]) * 0.5
        first = torch.stack([p[:, 0], torch.where(along_u, ma, p[:, 1]), torch.where(along_u, p[:, 2], ma), mb], 1)
        second = torch.stack([ma, torch.where(along_u, p[:, 1], mb), torch.where(along_u, mb, p[:, 2]), p[:, 3]], 1)
        mu, mv = (uv[:, :1] + uv[:, 1:2]) * 0.5, (uv[:, 2:3] + uv[:, 3:]) * 0.5
        uv1 = torch.where(along_u, torch.cat([uv[:, :1], mu, uv[:, 2:]], 1), torch.cat([uv[:, :3], mv], 1))
        uv2 = torch.where(along_u, torch.cat([mu, uv[:, 1:]], 1), torch.cat([uv[:, :2], mv, uv[:, 3:]], 1))
        ray, p, uv = ray.repeat(2), torch.cat([first, second]), torch.cat([uv1, uv2])


def exact(case, seed):
    """Hits on the terrain in 64 bits.  The other scenes' images and hits have no such value here: their sampling
    decisions, and the extraction of subdivision surfaces, would have to be the library's own."""
    if case["scene"] != "terrain" or case["kind"] not in ("rays", "world"):
        return None
    dev = torch.device("cuda", torch.cuda.current_device()) if torch.cuda.is_available() else torch.device("cpu")
    rays = _terrain_rays(case, seed, dev)
    P = torch.tensor(_terrain_patches(case["grid"], seed), dtype=torch.float64, device=dev)
    n = rays.shape[1]
    t = torch.full((n,), math.inf, dtype=torch.float64, device=dev)
    u, v, aux = (torch.zeros(n, dtype=torch.float64, device=dev) for _ in range(3))
    for a in range(0, n, 1 << 18):
        s = slice(a, min(n, a + (1 << 18)))
        w = rays[:, s].double()
        _trace64(P, case["grid"], case["dice_rate"], w, t[s], u[s], v[s], aux[s])
        # the rectangle light, met where the ray crosses its plane
        tl = (LIGHT_POS[2] - w[2]) / w[5]
        x, y = w[0] + w[3] * tl - LIGHT_POS[0], w[1] + w[4] * tl - LIGHT_POS[1]
        lit = (tl > 0) & (tl < t[s]) & (x.abs() <= LIGHT_SIZE / 2) & (y.abs() <= LIGHT_SIZE / 2)
        t[s] = torch.where(lit, tl, t[s])
        for q in (u, v, aux):
            q[s] = torch.where(lit, 0.0, q[s])
    out = {"t": t, "inst": None, "u": u, "v": v, "aux": aux}
    if case.get("shade"):
        out["records"] = None
    return out
