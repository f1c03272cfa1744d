"""The workloads this renderer is timed on, through its public entry points.

Every case is something a program using the framework does in earnest: ray
batches over a triangle soup (picking, occlusion baking, the traversal
benchmark), offline frames, progressive and tiled interactive frames, the
preview drawn while instances are edited, a frame rendered with a learned
guide trained from scratch, the guide network alone in both directions, and a
render server draining a queue of jobs.

    listed()             the cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what the program holds before the call
    run(state)           one pass
    work(case)           bytes and flops the pass cannot do without
    tolerance(case)      how far another correct implementation may be off
    exact(case, seed)    the same outputs in 64 bits, without this package
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from lavaframe_amd import lfh, scenes

GUIDE_LO, GUIDE_HI = (0.0, 0.0, 0.0), (6.0, 3.0, 4.0)   # the guiding room's box


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # a picking / probing query of a host program: a handful of rays, latency only
        {"name": "pick_1k", "kind": "closest", "tris": 20000, "rays": 1021, "pattern": "incoherent", "bvh": "sah"},
        # the traversal benchmark: 4096 x 2048 pinhole rays and as many incoherent ones, 1M triangles
        {"name": "closest_16m", "kind": "closest", "tris": 1048576, "rays": 16777216, "pattern": "mixed",
         "bvh": "sah"},
        # occlusion baking over a scene whose BVH the device built: an odd number of incoherent rays
        {"name": "occlusion_2m", "kind": "any", "tris": 700001, "rays": 2097143, "pattern": "incoherent",
         "bvh": "device"},
        # an offline frame of the Cornell box at the benchmark's size
        {"name": "cornell_64spp", "kind": "frame", "scene": "cornell", "width": 256, "height": 256, "depth": 4,
         "spp": 64},
        # an offline frame of the instanced outdoor scene (environment map, glass, metal): the largest
        {"name": "instanced_1080p", "kind": "frame", "scene": "instanced", "width": 1920, "height": 1080, "depth": 8,
         "spp": 8},
        # the interactive viewer after the camera stops: one pass and one displayed image per frame, deep paths
        {"name": "viewer_720p", "kind": "viewer", "scene": "room", "width": 1280, "height": 720, "depth": 10,
         "tile": 0, "frames": 4},
        # the same viewer with tiles, as the reference draws: ragged tiles, many small passes, texture maps
        {"name": "tiles_400", "kind": "viewer", "scene": "textured", "width": 400, "height": 300, "depth": 4,
         "tile": 128, "frames": 2},
        # instances dragged in the editor: transforms re-uploaded, the preview redrawn at half size
        {"name": "edit_preview", "kind": "edit", "instances": 200, "width": 960, "height": 540, "scale": 0.5},
        # a guided frame from scratch: a new guide trained online while 24 passes render
        {"name": "guided_360p", "kind": "guided", "width": 640, "height": 360, "depth": 10, "spp": 24},
        # the guide network alone, device-resident queries
        {"name": "guide_1m", "kind": "guide_forward", "queries": 1048576},
        # its loss and gradient over one optimisation batch
        {"name": "guide_grad_64k", "kind": "guide_grad", "queries": 65536},
        # a render server draining small jobs of several scenes and sizes
        {"name": "serve_6", "kind": "serve", "jobs": 6, "width": 320, "height": 180, "spp": 16},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["closest", "closest", "any", "frame", "frame", "viewer", "viewer", "edit", "guided",
                       "guide_forward", "guide_grad", "serve"])
    if kind in ("closest", "any"):
        return {"kind": kind, "tris": _log_int(rng, 1000, 1000000), "rays": _log_int(rng, 500, 12000000) | 1,
                "pattern": rng.choice(["incoherent", "pinhole", "mixed"]), "bvh": rng.choice(["sah", "device"])}
    if kind == "frame":
        scene = rng.choice(["cornell", "instanced", "room", "textured"])
        w = _log_int(rng, 64, 1400)
        return {"kind": kind, "scene": scene, "width": w, "height": max(16, int(w * rng.uniform(0.4, 1.0))),
                "depth": rng.randint(2, 10), "spp": rng.randint(1, 8 if w > 600 else 48)}
    if kind == "viewer":
        w = _log_int(rng, 64, 1280)
        h = max(16, int(w * rng.uniform(0.4, 1.0)))
        return {"kind": kind, "scene": rng.choice(["cornell", "room", "textured", "instanced"]), "width": w,
                "height": h, "depth": rng.randint(2, 10),
                "tile": rng.choice([0, 0, max(32, w // rng.randint(2, 5))]), "frames": rng.randint(1, 4)}
    if kind == "edit":
        w = _log_int(rng, 160, 1920)
        return {"kind": kind, "instances": _log_int(rng, 20, 600), "width": w, "height": max(90, w * 9 // 16),
                "scale": rng.choice([0.25, 0.5, 0.75, 1.0])}
    if kind == "guided":
        w = _log_int(rng, 160, 960)
        return {"kind": kind, "width": w, "height": max(90, w * 9 // 16), "depth": rng.randint(4, 10),
                "spp": rng.randint(5, 24)}
    if kind == "guide_forward":
        return {"kind": kind, "queries": _log_int(rng, 1000, 4000000)}
    if kind == "guide_grad":
        return {"kind": kind, "queries": _log_int(rng, 500, 65536)}
    w = _log_int(rng, 64, 640)
    return {"kind": kind, "jobs": rng.randint(1, 10), "width": w, "height": max(36, w * 9 // 16),
            "spp": rng.randint(2, 24)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _soup_vertices(n, seed):
    """n equilateral triangles (n, 3, 3): centres U[0,1]^3, random rotation, edge U(0.002, 0.02)."""
    g = _gen(seed)
    c = torch.rand(n, 1, 3, generator=g, device="cuda", dtype=torch.float64)
    edge = 0.002 + 0.018 * torch.rand(n, 1, 1, generator=g, device="cuda", dtype=torch.float64)
    a = torch.randn(n, 3, generator=g, device="cuda", dtype=torch.float64)
    b = torch.randn(n, 3, generator=g, device="cuda", dtype=torch.float64)
    a = a / a.norm(dim=1, keepdim=True)
    b = b - (a * b).sum(1, keepdim=True) * a
    b = b / b.norm(dim=1, keepdim=True)
    ang = [math.radians(d) for d in (90.0, 210.0, 330.0)]
    v = torch.stack([(math.cos(t) * a + math.sin(t) * b) / math.sqrt(3.0) for t in ang], 1)
    return (v * edge + c).to(torch.float32)


def _rays(n, pattern, seed):
    """(n, 8) float32 on the device: origin, tmin, direction, tmax."""
    g = _gen(seed + 7919)
    r = torch.empty(n, 8, device="cuda")
    r[:, 3] = 0.0
    r[:, 7] = scenes.RAY_TMAX
    coherent = {"pinhole": n, "incoherent": 0, "mixed": n // 2}[pattern]
    if coherent:
        h = max(1, int(math.sqrt(coherent / 2)))
        w = (coherent + h - 1) // h
        # the benchmark's camera, moved a little by the seed
        eye = (0.5 + 0.01 * (seed % 7), 0.5, -1.5)
        pos, rt, up, fw = (torch.tensor(x, device="cuda", dtype=torch.float64)
                           for x in scenes.camera_basis(eye, (0.5, 0.5, 0.5)))
        k = torch.arange(coherent, device="cuda")
        scale = math.tan(math.radians(40.0) * 0.5)
        x = (((k % w).double() + 0.5) / w * 2 - 1) * scale
        y = ((torch.div(k, w, rounding_mode="floor").double() + 0.5) / h * 2 - 1) * scale * h / w
        d = x[:, None] * rt + y[:, None] * up + fw
        r[:coherent, 0:3] = pos.float()
        r[:coherent, 4:7] = (d / d.norm(dim=1, keepdim=True)).float()
    if coherent < n:
        m = n - coherent
        r[coherent:, 0:3] = torch.rand(m, 3, generator=g, device="cuda")
        d = torch.randn(m, 3, generator=g, device="cuda")
        r[coherent:, 4:7] = d / d.norm(dim=1, keepdim=True)
    return r


def _guide_inputs(n, seed):
    """(n, 9) positions in the room, normals, outgoing directions in the normal's hemisphere."""
    g = _gen(seed + 104729)
    lo, hi = (torch.tensor(v, device="cuda") for v in (GUIDE_LO, GUIDE_HI))
    x = torch.empty(n, 9, device="cuda")
    x[:, 0:3] = lo + (hi - lo) * torch.rand(n, 3, generator=g, device="cuda")
    for k in (3, 6):
        d = torch.randn(n, 3, generator=g, device="cuda")
        x[:, k:k + 3] = d / d.norm(dim=1, keepdim=True)
    flip = (x[:, 3:6] * x[:, 6:9]).sum(1, keepdim=True) < 0
    x[:, 6:9] = torch.where(flip, -x[:, 6:9], x[:, 6:9])
    return x


def _guide_targets(n, seed):
    """Directions gathered around a few lights, and their long-tailed weights."""
    g = _gen(seed + 1299709)
    c = torch.randn(4, 3, generator=g, device="cuda")
    d = c[torch.randint(0, 4, (n,), generator=g, device="cuda")] + 0.5 * torch.randn(n, 3, generator=g, device="cuda")
    return d / d.norm(dim=1, keepdim=True), torch.rand(n, generator=g, device="cuda").pow(4) * 5.0


def _guide_params(seed):
    """Parameters of a partly trained guide: the initial scale, outputs of order one."""
    p = np.random.default_rng(seed + 15485863).uniform(-1, 1, lfh.Guide.N_PARAMS).astype(np.float32)
    return p * np.float32(0.3)


# The scenes of the frame, viewer and server cases are assets: the program has
# loaded them, each seed renders other random-number frames of them.
@functools.lru_cache(maxsize=None)
def _asset(name):
    if name == "cornell":
        return scenes.cornell()
    if name == "room":
        return scenes.aperture_room()
    if name == "textured":
        return scenes.textured_room()
    return scenes.instanced(n_meshes=24, n_instances=400, max_tris=60000, hdr_size=(1024, 512))


@functools.lru_cache(maxsize=4)
def _edit_asset(instances):
    return scenes.instanced(n_meshes=12, n_instances=instances, max_tris=20000, hdr_size=(256, 128), light_count=4,
                            build=False)


@functools.lru_cache(maxsize=None)
def _stream():
    """The one stream a program's ray batches run on."""
    return torch.cuda.Stream()


def _render_options(case, seed):
    tile = case.get("tile", 0)
    return dict(width=case["width"], height=case["height"], tile_width=tile or case["width"],
                tile_height=tile or case["height"], max_depth=case.get("depth", 4), frame_offset=1 + seed % 100000)


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "case": case}
    if kind in ("closest", "any"):
        scene = lfh.Scene()
        scene.add_material(lfh.MATERIAL_DEFAULT)
        scene.add_instance(scene.add_mesh(_soup_vertices(case["tris"], seed).cpu().numpy()), None, 0)
        scene.build() if case["bvh"] == "sah" else scene.flatten()
        ctx = s["ctx"] = lfh.Context.from_scene(scene, width=16, height=16, tile_width=16, tile_height=16)
        ctx.set_stream(_stream().cuda_stream)
        n = s["n"] = case["rays"]
        s["rays"] = _rays(n, case["pattern"], seed)
        if kind == "closest":
            hits = s["hits"] = torch.zeros(n, 6, device="cuda", dtype=torch.int32)
            s["out"] = {"ids": hits[:, 0:3], "tuv": hits.view(torch.float32)[:, 3:6]}
        else:
            s["out"] = s["hits"] = torch.zeros(n, device="cuda", dtype=torch.uint8)
    elif kind in ("frame", "viewer"):
        scene = _asset(case["scene"])
        s["ctx"] = lfh.Context.from_scene(scene, **_render_options(case, seed))
        s["cam"] = scene.camera()
        s["pp"] = lfh.Postprocess.make(tonemap_index=2)
    elif kind == "edit":
        scene = _edit_asset(case["instances"])
        s["ctx"] = lfh.Context.from_scene(scene, device_bvh=True, **_render_options(case, seed))
        s["cam"] = scene.camera()
        t = scene.arrays()["transforms"].copy()
        rng = np.random.default_rng(seed)
        t[:-1, 12:15] += rng.normal(0.0, 0.5, (len(t) - 1, 3)).astype(np.float32)   # all but the floor
        s["transforms"] = t
    elif kind == "guided":
        scene = _asset("room")
        s["ctx"] = lfh.Context.from_scene(scene, estimator=1, guiding=1, **_render_options(case, seed))
        s["cam"] = scene.camera()
        s["seed"] = seed
    elif kind == "guide_forward":
        s["guide"] = lfh.Guide(GUIDE_LO, GUIDE_HI)
        s["guide"].set_params(_guide_params(seed))
        s["x"] = _guide_inputs(case["queries"], seed)
        s["out"] = torch.zeros(case["queries"], 40, device="cuda")
    elif kind == "guide_grad":
        s["guide"] = lfh.Guide(GUIDE_LO, GUIDE_HI)
        s["guide"].set_params(_guide_params(seed))
        d, w = _guide_targets(case["queries"], seed)
        s["x"], s["d"], s["w"] = (v.cpu().numpy() for v in (_guide_inputs(case["queries"], seed), d, w))
    else:
        s["server"] = lfh.Server(budget_bytes=32 << 30)
        jobs = s["jobs"] = []
        for k in range(case["jobs"]):
            # sizes and sample counts of a mixed queue, the largest first submitted last
            f = (0.35, 0.6, 1.0)[k % 3]
            w, h = max(16, int(case["width"] * f) | 1), max(16, int(case["height"] * f))
            jobs.append((_asset(("cornell", "room", "textured")[k % 3]), max(1, case["spp"] >> (k % 3)),
                         dict(width=w, height=h, tile_width=w, tile_height=h, frame_offset=1 + (seed + 37 * k) % 100000)))
    torch.cuda.synchronize()   # the inputs are in hand
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "closest":
        s["ctx"].trace_closest_device(s["rays"].data_ptr(), s["n"], s["hits"].data_ptr())
        return s["out"]
    if kind == "any":
        s["ctx"].trace_any_device(s["rays"].data_ptr(), s["n"], s["hits"].data_ptr())
        return s["out"]
    if kind == "frame":
        ctx = s["ctx"]
        ctx.update(s["cam"], reset=True)
        ctx.render_passes(case["spp"])
        return ctx.output_hdr()
    if kind == "viewer":
        ctx = s["ctx"]
        tiles = 1
        if case["tile"]:
            tiles = math.ceil(case["width"] / min(case["tile"], case["width"])) * \
                math.ceil(case["height"] / min(case["tile"], case["height"]))
        ctx.update(s["cam"], reset=True)
        for _ in range(case["frames"]):
            for _ in range(tiles):
                ctx.update(s["cam"])
                ctx.render()
            ldr = ctx.output_ldr(s["pp"])
        return {"ldr": ldr, "hdr": ctx.output_hdr()}
    if kind == "edit":
        ctx = s["ctx"]
        ctx.update_instances(transforms=s["transforms"])
        ctx.update(s["cam"], reset=True)
        return ctx.render_preview(case["scale"])
    if kind == "guided":
        ctx = s["ctx"]
        guide = lfh.Guide(GUIDE_LO, GUIDE_HI, seed=s["seed"], lr=1.5e-3)
        ctx.set_guide(guide, train_every=1)
        ctx.update(s["cam"], reset=True)
        ctx.render_passes(case["spp"])
        out = {"hdr": ctx.output_hdr(), "params": guide.params()}
        ctx.set_guide(None)
        guide.close()
        return out
    if kind == "guide_forward":
        s["guide"].forward_device(s["x"].data_ptr(), case["queries"], s["out"].data_ptr(),
                                  torch.cuda.current_stream().cuda_stream)
        return s["out"]
    if kind == "guide_grad":
        loss, grad = s["guide"].loss_grad(s["x"], s["d"], s["w"])
        return {"loss": loss, "grad": grad}
    srv = s["server"]
    ids = [(srv.submit_scene(scene, spp, **opt), opt) for scene, spp, opt in s["jobs"]]
    srv.run_until_idle()
    out = [srv.result(i, opt["width"], opt["height"]) for i, opt in ids]
    for i, _ in ids:
        srv.release(i)
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
_SCENE_TRIS = {"cornell": 34, "room": 197000, "textured": 26, "instanced": 300000}


def _ray_flops(tris):
    """One ray: two boxes (24 flops each) on each level of a binary tree, two triangle tests (60 flops)."""
    return 48.0 * math.log2(tris + 2) + 120.0


def _path_flops(tris, depth):
    """One sample: an extension and a shadow ray and one shading (about 500 flops) per vertex, Russian roulette
    ending paths after about four vertices."""
    return min(depth, 4) * (2.0 * _ray_flops(tris) + 500.0)


def work(case):
    kind = case["kind"]
    if kind in ("closest", "any"):
        return {"bytes": case["rays"] * (32.0 + (24.0 if kind == "closest" else 1.0)) + case["tris"] * 36.0,
                "flops": case["rays"] * _ray_flops(case["tris"])}
    if kind in ("frame", "viewer"):
        tris, pix = _SCENE_TRIS[case["scene"]], case["width"] * case["height"]
        n = case["spp"] if kind == "frame" else case["frames"]
        return {"bytes": tris * 60.0 + pix * (12.0 if kind == "frame" else 12.0 + 3.0 * n),
                "flops": n * pix * _path_flops(tris, case["depth"])}
    if kind == "edit":
        pix = int(case["width"] * case["scale"]) * int(case["height"] * case["scale"])
        return {"bytes": pix * 12.0 + case["instances"] * 64.0 + 40000 * 60.0,
                "flops": pix * _path_flops(40000, 2)}
    if kind == "guided":
        pix = case["width"] * case["height"]
        n = float(pix * case["spp"])
        return {"bytes": pix * 12.0 + 197000 * 60.0,
                "flops": n * (_path_flops(197000, case["depth"]) + min(case["depth"], 4) * 29696.0)
                + 64 * 65536 * 3 * 29696.0}
    if kind == "guide_forward":
        return {"bytes": case["queries"] * 196.0, "flops": case["queries"] * 29696.0}
    if kind == "guide_grad":
        return {"bytes": case["queries"] * 52.0 + 60320.0, "flops": case["queries"] * 3 * 29696.0}
    flops = bytes_ = 0.0
    for k in range(case["jobs"]):
        f = (0.35, 0.6, 1.0)[k % 3]
        pix = int(case["width"] * f) * int(case["height"] * f)
        tris = _SCENE_TRIS[("cornell", "room", "textured")[k % 3]]
        flops += max(1, case["spp"] >> (k % 3)) * pix * _path_flops(tris, 4)
        bytes_ += pix * 12.0 + tris * 60.0
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind in ("closest", "any"):
        # the same hits, bit for bit (two BVHs of one soup: no difference in 35M rays), save
        # for a ray that grazes a triangle so flatly that Moller-Trumbore's own t is off by
        # more than 1/1024
        return {"rel": 1e-5, "max": 0.99, "differ": 1e-6}
    if kind == "guide_forward":
        return {"rel": 1e-2, "max": 0.3}    # bf16 operands, fp32 sums: 0.0043 off the 64-bit network
    if kind == "guide_grad":
        return {"rel": 2e-2, "max": 0.5}    # the same through the backward products: 0.0074
    if kind == "guided":
        return {"rel": 1e-2, "max": 0.99}   # training carries a rounding on to every later pass
    # another fp32 implementation of these images is off by 1e-8 to 2.5e-5 as a whole and by up
    # to 0.007 of the rms at a pixel; a path that meets a last-bit difference of sin or pow at a
    # branch goes another way, and a small image shows one such path
    return {"rel": 1e-3, "max": 0.99, "differ": 1e-3}


# ---------------------------------------------------------------------------
# the same outputs in 64 bits
# ---------------------------------------------------------------------------
def _exact_closest(case, seed):
    if case["tris"] * case["rays"] > 2e10:
        return None   # brute force over all pairs
    v = _soup_vertices(case["tris"], seed).double()
    v0, e0, e1 = v[:, 0], v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]
    n = torch.linalg.cross(e0, e1)
    r = _rays(case["rays"], case["pattern"], seed).double()
    out = torch.zeros(case["rays"], 3, device="cuda", dtype=torch.float64)
    step = max(1, int(4e7) // case["tris"])
    inf = float("inf")
    for k in range(0, case["rays"], step):
        o, d = r[k:k + step, None, 0:3], r[k:k + step, None, 4:7]
        # det = e0 . (d x e1) = -d . n and, with tv = o - v0 and q = tv x d:
        # u det = e1 . q, v det = -e0 . q, t det = tv . n
        det = -(d * n).sum(-1)
        tv = o - v0
        q = torch.linalg.cross(tv, d.expand_as(tv))
        u, w = (e1 * q).sum(-1) / det, -(e0 * q).sum(-1) / det
        t = (tv * n).sum(-1) / det
        ok = (u >= 0) & (w >= 0) & (u + w <= 1) & (t >= 0)
        best, i = torch.where(ok, t, torch.full_like(t, inf)).min(1)
        hit = best < scenes.RAY_TMAX
        rows = torch.arange(len(i), device="cuda")
        zero = torch.zeros_like(best)
        out[k:k + step, 0] = torch.where(hit, best, torch.full_like(best, scenes.RAY_TMAX))
        out[k:k + step, 1] = torch.where(hit, u[rows, i], zero)
        out[k:k + step, 2] = torch.where(hit, w[rows, i], zero)
    return {"ids": None, "tuv": out}


def _exact_guide(params, x):
    lo, hi = (torch.tensor(v, device="cuda", dtype=torch.float64) for v in (GUIDE_LO, GUIDE_HI))
    p, n, wo = ((x[:, 0:3] - lo) / (hi - lo)).clamp(0, 1), x[:, 3:6], x[:, 6:9]
    f = []
    for src, octaves in ((p, 6), (n, 2), (wo, 2)):
        for a in range(3):
            for k in range(octaves):
                f += [torch.sin(2.0 ** k * math.pi * src[:, a]), torch.cos(2.0 ** k * math.pi * src[:, a])]
    y = torch.stack(f + [wo[:, 0], wo[:, 1], wo[:, 2], torch.ones_like(wo[:, 0])], 1)
    at = 0
    for k, width in enumerate((64, 64, 64, 40)):
        y = y @ params[at:at + 64 * width].view(64, width) + params[at + 64 * width:at + 65 * width]
        at += 65 * width
        if k < 3:
            y = y.clamp_min(0)
    return y


def exact(case, seed):
    kind = case["kind"]
    if kind == "closest":
        return _exact_closest(case, seed)
    if kind == "guide_forward":
        params = torch.from_numpy(_guide_params(seed)).cuda().double()
        x = _guide_inputs(case["queries"], seed).double()
        return torch.cat([_exact_guide(params, c) for c in x.split(1 << 18)])
    if kind == "guide_grad":
        params = torch.from_numpy(_guide_params(seed)).cuda().double().requires_grad_(True)
        d, w = (v.double() for v in _guide_targets(case["queries"], seed))
        o = _exact_guide(params, _guide_inputs(case["queries"], seed).double()).view(-1, 8, 5)
        mu = o[..., 0:3] / o[..., 0:3].norm(dim=-1, keepdim=True)
        kappa = o[..., 3].clamp(-3, 7).exp()
        logp = torch.logsumexp(torch.log_softmax(o[..., 4], 1)
                               + torch.log(kappa / (2 * math.pi * -torch.expm1(-2 * kappa)))
                               + kappa * ((mu * d[:, None]).sum(-1) - 1), 1)
        loss = -(w * logp).mean()
        loss.backward()
        return {"loss": float(loss.detach()), "grad": params.grad}
    # occlusion is a byte; a path-traced image is a sum over chains of discrete
    # decisions (lobe, roulette, hit or miss), each taken on 32-bit values, that
    # a 64-bit restatement takes differently now and then: no such value
    return None
