"""The framework's work as its users ask for it, for measuring: path-traced
frames (the headline interior, interactive previews, every family of scene the
framework ships), a batch of scenes, one step of inverse rendering, and ray
queries.  listed() names fixed cases, draw() makes more of the same ranges.

A case of kind
  frame    one ymrt_render_frame (Scene.render_frame) of a resident scene:
           the next progressive frame of a still.  "post": followed by
           accumulate and tonemap, as an interactive view does per frame.
           "noalloc": through Scene.render_frame_noalloc.
  batch    one Context.render_batch over several scenes of unlike size
  inverse  autograd.render, a mean-square loss and its backward pass
  rays     Scene.trace_closest or Scene.trace_any over rays in device memory
"""
import math

import numpy as np
import torch

import ymrt_amd
from ymrt_amd import abi, autograd, scenes

_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        _ctx = ymrt_amd.Context(0)
    return _ctx


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest frame in use: a thumbnail of a Cornell box, where
        # launches and near-empty passes are the time
        dict(name="thumbnail_cornell_256_1spp", kind="frame", scene="cornell", width=256, height=256, spp=1,
             depth=8, sampler="halton"),
        # a frame for callers that cannot allocate, in the framework's fixed
        # scratch memory: PCG samples, analytic sphere and sphere light,
        # Russian roulette, odd sizes
        dict(name="noalloc_sphere_317x241_8spp", kind="frame", scene="cornell_sphere", width=317, height=241, spp=8,
             depth=6, sampler="pcg", rr=1, noalloc=True),
        # one frame of an interactive view: 1 sample per pixel, accumulated
        # and tonemapped
        dict(name="preview_interior_1080p_1spp", kind="frame", scene="interior", width=1920, height=1080, spp=1,
             depth=8, sampler="halton", post=True),
        # the headline workload of the benchmark: a full-quality frame
        dict(name="final_interior_1080p_64spp", kind="frame", scene="interior", width=1920, height=1080, spp=64,
             depth=8, sampler="halton"),
        # sun and sky geometry: distant light, analytic spheres, glass, a fog
        # box that shadow rays cross; odd image size
        dict(name="outdoor_fog_1279x719_8spp", kind="frame", scene="outdoor", width=1279, height=719, spp=8, depth=6,
             sampler="halton"),
        # materials from procedural texture graphs, normal and bump maps
        dict(name="procedural_box_640x480_16spp", kind="frame", scene="textured", width=640, height=480, spp=16,
             depth=6, sampler="halton"),
        # a heterogeneous medium (voxel grid) inside a Cornell box
        dict(name="smoke_cornell_512_16spp", kind="frame", scene="media", width=512, height=512, spp=16, depth=8,
             sampler="halton"),
        # many views and scenes rendered together, a dataset's worth of small
        # and middling frames
        dict(name="batch_24_scenes", kind="batch", count=24, min_tris=1000, max_tris=100000, max_res=512, max_spp=16,
             depth=6),
        # one optimisation step of inverse rendering: 256^2 texels, 8
        # roughnesses, 64^3 densities and 3 albedos
        dict(name="inverse_cornell_512_16spp", kind="inverse", size=512, spp=16, depth=6, texels=256, grid=64),
        # incoherent closest-hit rays against 2 M triangles
        dict(name="rays_closest_4M_2Mtri", kind="rays", any=False, scene="heightfield", side=1001, rays=1 << 22),
        # visibility segments, a ragged count, half a million triangles
        dict(name="rays_any_1000003_500ktri", kind="rays", any=True, scene="heightfield", side=501, rays=1000003),
        # a few rays, as picking and collision queries ask
        dict(name="rays_closest_4095_cornell", kind="rays", any=False, scene="cornell", side=0, rays=4095),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "rays", "rays", "batch", "inverse"])
    if kind == "rays":
        field = rng.random() < 0.7
        return dict(kind="rays", any=rng.random() < 0.5, scene="heightfield" if field else "cornell",
                    side=_log(rng, 17, 1001) if field else 0, rays=_log(rng, 1000, 1 << 22))
    if kind == "batch":
        return dict(kind="batch", count=rng.randint(2, 32), min_tris=1000, max_tris=_log(rng, 2000, 200000),
                    max_res=rng.choice([256, 512]), max_spp=rng.choice([4, 16]), depth=rng.randint(2, 8))
    if kind == "inverse":
        return dict(kind="inverse", size=_log(rng, 48, 512), spp=_log(rng, 1, 16), depth=rng.randint(2, 6),
                    texels=_log(rng, 16, 256), grid=_log(rng, 8, 64))
    scene = rng.choice(["cornell", "cornell_sphere", "interior", "interior", "outdoor", "textured", "media"])
    width = _log(rng, 96, 1920)
    height = max(64, int(width * rng.uniform(0.5, 1.0)))
    most = max(1, min(64, 40000000 // (width * height)))
    spp = _log(rng, 1, most)
    # the fixed memory holds 65536 paths at a time: small frames go there
    noalloc = width * height * spp <= 2000000 and rng.random() < 0.3
    return dict(kind="frame", scene=scene, width=width, height=height, spp=spp, depth=rng.randint(2, 10),
                sampler=rng.choice(["halton", "halton", "pcg"]), rr=int(rng.random() < 0.25),
                post=rng.random() < 0.3, noalloc=noalloc)


# ------------------------------------------------------------------- scenes
def _noise_texture(n, rng, octaves=4):
    """RGBA8 value noise of n x n texels: random lattices, enlarged and summed."""
    acc = torch.zeros((1, 3, n, n), dtype=torch.float32, device="cuda")
    for o in range(octaves):
        cells = 16 * 2 ** o
        lat = torch.from_numpy(rng.random((1, 3, cells, cells), np.float32)).cuda()
        acc += 0.5 ** o * torch.nn.functional.interpolate(lat, size=(n, n), mode="bilinear", align_corners=False)
    acc = (acc - acc.amin()) / (acc.amax() - acc.amin())
    tex = np.full((n, n, 4), 255, np.uint8)
    tex[..., :3] = (acc[0].permute(1, 2, 0) * 255.0).round().to(torch.uint8).cpu().numpy()
    return tex


def _interior(width, height, rng):
    """scenes.interior with 2048^2 textures and instance positions from rng."""
    sa = scenes.interior(width, height, tex_size=64, halton_seed=int(rng.integers(1 << 31)))
    for t in sa.textures:
        t["texels"] = _noise_texture(2048, rng)
    for it in sa.instances[:40]:
        o2w = it["o2w"].copy()
        o2w[:3, 3] += rng.uniform(-0.4, 0.4, 3).astype(np.float32) * np.float32([1.0, 0.3, 1.0])
        it["o2w"] = o2w
        w2o = np.linalg.inv(o2w.astype(np.float64)).astype(np.float32)
        w2o[3, :] = (0.0, 0.0, 0.0, 1.0)
        it["w2o"] = w2o
    return sa


def _arrays(name, width, height, rng):
    seed = int(rng.integers(1 << 31))
    if name == "interior":
        sa = _interior(width, height, rng)
    elif name == "cornell":
        sa = scenes.cornell_box(width, height, halton_seed=seed)
    elif name == "cornell_sphere":
        sa = scenes.cornell_box(width, height, halton_seed=seed, analytic_sphere=True, sphere_light=True)
    elif name == "outdoor":
        sa = scenes.outdoor(width, height, fog=True, halton_seed=seed)
    elif name == "textured":
        sa = scenes.textured_box(width, height, halton_seed=seed)
    elif name == "media":
        sa = scenes.cornell_media(width, height, grid=True, halton_seed=seed, sigma=4.0)
        sa.grids[0] = rng.random(sa.grids[0].shape, np.float32)
    else:
        raise ValueError(name)
    # every seed sees the scene from a place of its own
    p = np.asarray(sa.camera["position"], np.float32) + rng.uniform(-0.05, 0.05, 3).astype(np.float32)
    sa.camera["position"] = tuple(p.tolist())
    return sa


def _settings(case):
    name = case["scene"]
    return abi.render_settings(case["width"], case["height"], case["spp"], case["depth"],
                               sampler=abi.SAMPLER_HALTON if case["sampler"] == "halton" else abi.SAMPLER_PCG,
                               volume=int(name in ("interior", "outdoor", "media")),
                               distant_light=int(name == "outdoor"), rr=int(case.get("rr", 0)))


def _batch_work(case, rng):
    """[(triangles, resolution, spp)] of a batch: unlike frames, as drawn from
    a data set."""
    res = [r for r in (128, 256, 512) if r <= case["max_res"]]
    spp = [s for s in (1, 4, 16) if s <= case["max_spp"]]
    out = []
    for _ in range(case["count"]):
        t = math.exp(rng.uniform(math.log(case["min_tris"]), math.log(case["max_tris"])))
        out.append((int(t), int(rng.choice(res)), int(rng.choice(spp))))
    return out


def _batch_sizes(case):
    """The frame sizes of a batch case: the same for every seed."""
    return _batch_work(case, np.random.default_rng(17 + case["count"]))


# ------------------------------------------------------------- prepare, run
def prepare(case, seed):
    rng = np.random.default_rng(seed)
    ctx = _context()
    if case["kind"] == "frame":
        w, h = case["width"], case["height"]
        s = dict(kind="frame", scene=ymrt_amd.Scene(ctx, _arrays(case["scene"], w, h, rng)), rs=_settings(case),
                 frame=1 + int(rng.integers(64)), noalloc=bool(case.get("noalloc")),
                 noise=torch.empty((h, w, 4), dtype=torch.float32, device="cuda"))
        if case.get("post"):
            # the running mean of the frames before this one
            s["accum"] = torch.from_numpy(rng.gamma(1.0, 0.5, (h, w, 4)).astype(np.float32)).cuda()
            s["accum"][..., 3] = 1.0
            s["view"] = torch.empty_like(s["accum"])
        return s
    if case["kind"] == "batch":
        jobs = []
        for tris, res, spp in _batch_sizes(case):
            sa = scenes.batch_scene(tris, res, res, int(rng.integers(1 << 31)))
            jobs.append((ymrt_amd.Scene(ctx, sa), abi.render_settings(res, res, spp, case["depth"]),
                         1 + int(rng.integers(64))))
        return dict(kind="batch", jobs=jobs)
    if case["kind"] == "inverse":
        n = case["size"]
        true = scenes.inverse_params(case["texels"], case["grid"], 8, int(rng.integers(1 << 20)))
        sa, targets = scenes.cornell_inverse(n, n, true, halton_seed=int(rng.integers(1 << 31)))
        scene = ymrt_amd.Scene(ctx, sa)
        rs = abi.render_settings(n, n, case["spp"], case["depth"], volume=1)
        frame = 1 + int(rng.integers(64))
        photo = scene.render_frame(rs, frame + 1)[0][..., :3].contiguous()
        guess = scenes.perturb_params(true, 0.3, int(rng.integers(1 << 20)))
        albedo = rng.uniform(0.2, 0.8, (len(targets["albedo"]), 3)).astype(np.float32)
        leaf = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda().requires_grad_()  # noqa: E731
        return dict(kind="inverse", scene=scene, rs=rs, frame=frame, targets=targets, photo=photo,
                    params=dict(albedo=leaf(albedo), roughness=leaf(guess["roughness"]),
                                texture=leaf(guess["texture"]), density=leaf(guess["density"])))
    sa = _ray_scene(case, seed)
    closest, shadow = scenes.stress_rays(sa, case["rays"], seed % 1000003, seed % 1000003 + 1, seed % 1000003 + 2)
    return dict(kind="rays", any=case["any"], scene=ymrt_amd.Scene(ctx, sa),
                rays=ymrt_amd.Scene.rays_to_device(shadow if case["any"] else closest))


def _ray_scene(case, seed):
    if case["scene"] == "heightfield":
        return scenes.heightfield(case["side"], seed=1 + seed % 1000003)
    return scenes.cornell_box(64, 64, halton_seed=seed % 1000003)


def run(s):
    if s["kind"] == "frame":
        if s["noalloc"]:
            s["scene"].render_frame_noalloc(s["rs"], s["frame"], s["noise"])
        else:
            s["scene"].render_frame(s["rs"], s["frame"], s["noise"])
        if "accum" not in s:
            return s["noise"]
        ymrt_amd.accumulate(s["noise"], s["accum"], 4)
        s["view"].copy_(s["accum"])
        ymrt_amd.tonemap(s["view"])
        return dict(noise=s["noise"], view=s["view"])
    if s["kind"] == "batch":
        return [img for img, _ in _context().render_batch(s["jobs"])]
    if s["kind"] == "inverse":
        p = s["params"]
        img = autograd.render(s["scene"], s["rs"], s["targets"], frame=s["frame"], **p)
        loss = torch.nn.functional.mse_loss(img, s["photo"])
        names = sorted(p)
        grads = torch.autograd.grad(loss, [p[k] for k in names])
        return dict(image=img.detach(), **{"grad_" + k: g for k, g in zip(names, grads)})
    if s["any"]:
        return s["scene"].trace_any(s["rays"])
    hits = s["scene"].trace_closest(s["rays"])
    return dict(t=hits[:, 0].view(torch.float32), ids=hits[:, 1:])


# ------------------------------------------------------------ what it takes
def _triangles(case):
    if case["kind"] == "rays":
        return 2 * (case["side"] - 1) ** 2 if case["scene"] == "heightfield" else 1000
    return dict(interior=260000, cornell=1000, cornell_sphere=40, outdoor=30, textured=100, media=1000)[case["scene"]]


# one segment through a binary tree over T triangles: about 2 log2 T box
# tests of 18 operations and two triangle tests of 60
def _segment_flops(tris):
    return 36.0 * math.log2(max(2, tris)) + 120.0


# one vertex: surface frame, BSDF, light sample, sampling a direction
_VERTEX_FLOPS = 400.0


def _frame_work(pixels, spp, depth, tris, texels=0):
    # per vertex one extension segment and one or two shadow segments; paths
    # keep about two thirds of the vertices that their depth allows
    vertices = pixels * spp * max(1.0, 0.65 * depth)
    return dict(bytes=16.0 * pixels + 36.0 * tris + 4.0 * texels,
                flops=vertices * (2.5 * _segment_flops(tris) + _VERTEX_FLOPS))


def work(case):
    if case["kind"] == "frame":
        px = case["width"] * case["height"]
        w = _frame_work(px, case["spp"], case["depth"], _triangles(case),
                        4 * 2048 * 2048 if case["scene"] == "interior" else 0)
        if case.get("post"):
            w["bytes"] += px * 48.0
            w["flops"] += px * 60.0
        return w
    if case["kind"] == "batch":
        parts = [_frame_work(r * r, s, case["depth"], t) for t, r, s in _batch_sizes(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    if case["kind"] == "inverse":
        px = case["size"] ** 2
        f = _frame_work(px, case["spp"], case["depth"], 40)
        params = case["texels"] ** 2 * 3 + case["grid"] ** 3 + 17
        # the frame and its replay, whose events cost about a vertex again
        return dict(bytes=16.0 * px * 2 + 8.0 * params, flops=2.5 * f["flops"])
    t = _triangles(case)
    return dict(bytes=case["rays"] * (36.0 if case["any"] else 48.0) + 36.0 * t,
                flops=case["rays"] * _segment_flops(t))


def tolerance(case):
    if case["kind"] == "rays":
        # hits do not depend on the tree but for ties (a ray through a shared
        # edge): the bar of the parity tests, 99.99 % of rays (trees of other
        # leaf sizes gave the same bits)
        return dict(rel=1e-5, max=4e-5, differ=1e-4)
    if case["kind"] == "inverse":
        # gradients are sums of float atomics, in an order of their own in
        # every run: two runs measured 3e-6 to 6e-6 apart, at most 9e-6 in one
        # value
        return dict(rel=2e-5, max=4e-5)
    # frames are deterministic, and trees of other leaf sizes gave the same
    # bits; room for a path of a pixel that takes another branch after a tie
    return dict(rel=2e-5, max=0.2)


# ------------------------------------------------------------ in 64 bits
def exact(case, seed):
    """Closest hits by trying every triangle in 64 bits, where that is quick;
    a path-traced image has no value that plain arithmetic could give."""
    if case["kind"] != "rays" or case["any"] or case["scene"] != "cornell" or case["rays"] > 100000:
        return None
    sa = _ray_scene(case, seed)
    closest, _ = scenes.stress_rays(sa, case["rays"], seed % 1000003, seed % 1000003 + 1, seed % 1000003 + 2)
    o, d = (torch.from_numpy(closest[k].astype(np.float64)) for k in ("o", "d"))
    d = d / d.norm(dim=1, keepdim=True)
    best = torch.full((len(o),), float(np.float32(1e36)), dtype=torch.float64)  # a ray that hits nothing
    for it in sa.instances:
        m = sa.meshes[it["mesh"]]
        p = torch.from_numpy(m["pos"].astype(np.float64)) @ torch.from_numpy(it["o2w"][:3, :3].astype(np.float64)).T
        p = p + torch.from_numpy(it["o2w"][:3, 3].astype(np.float64))
        for tri in m["pidx"]:
            a, b, c = (p[int(k)] for k in tri)
            e1, e2 = b - a, c - a
            h = torch.linalg.cross(d, e2.expand_as(d))
            det = h @ e1
            s = o - a
            u = (s * h).sum(1) / det
            q = torch.linalg.cross(s, e1.expand_as(s))
            v = (d * q).sum(1) / det
            t = (q @ e2) / det
            # a ray through a shared edge belongs to one of its triangles
            ok = (u >= -1e-9) & (v >= -1e-9) & (u + v <= 1.0 + 1e-9) & (t > 1e-7) & (det != 0.0) & (t < best)
            best = torch.where(ok, t, best)
    return dict(t=best, ids=None)

