"""GPU traversal parity: the HIP closest-hit / any-hit kernels against the CPU
restatement of ClosestHit / AnyHit (closest_hit.glsl, anyhit.glsl) on the
same flattened BVH and rays.  Bar: prim / instance / material ids and the
bits of t, u, v identical (ties to the lowest (instance, prim))."""
import numpy as np
import pytest

from lavaframe_amd import lfh, scenes
from oracle import native

pytestmark = pytest.mark.gpu


def aimed_rays(scene, n, seed=0):
    """Rays from random origins towards random triangle centroids."""
    v = scene.arrays()["vertices"][:, :3].reshape(-1, 3, 3)
    rng = np.random.default_rng(seed)
    tgt = v[rng.integers(0, len(v), n)].mean(1)
    r = scenes.incoherent_rays(n, seed=seed + 1)
    d = tgt - r["org"]
    r["dir"] = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    return r


def _ctx(scene):
    arr = scene.arrays()
    desc, keep = lfh.desc_from_arrays(arr)
    opts = scene.options()
    return lfh.Context(desc, opts), arr


def _compare(gh, oh):
    assert gh.shape == oh.shape
    for k in ("prim", "inst", "mat"):
        bad = np.nonzero(gh[k] != oh[k])[0]
        assert bad.size == 0, f"{k} differs on {bad.size} rays, first {bad[:5]}: {gh[bad[:3]]} vs {oh[bad[:3]]}"
    for k in ("t", "u", "v"):
        g = gh[k].view(np.uint32)
        o = oh[k].view(np.uint32)
        bad = np.nonzero(g != o)[0]
        assert bad.size == 0, f"{k} bits differ on {bad.size} rays: {gh[bad[:3]]} vs {oh[bad[:3]]}"


@pytest.mark.parametrize("ntri,nray", [(1, 4096), (10, 20000), (10000, 200000)])
def test_soup_closest_and_any(ntri, nray):
    print(f"[trace] soup ntri={ntri} nray={nray}", flush=True)
    sc = scenes.soup(ntri, seed=ntri)
    ctx, arr = _ctx(sc)
    orc = native.OracleScene(arr)
    rays = np.concatenate([scenes.incoherent_rays(nray // 2, seed=3),
                           scenes.pinhole_rays(64, nray // 4 // 64), aimed_rays(sc, nray // 4, seed=6)])
    gh = ctx.trace_closest(rays)
    oh = orc.trace_closest(rays, tie_mode=1)
    _compare(gh, oh)
    assert (gh["prim"] >= 0).sum() > nray // 20
    occ = ctx.trace_any(rays)
    oocc = orc.trace_any(rays)
    assert np.array_equal(occ, oocc)
    # any-hit must agree with closest-hit over the same interval
    assert np.array_equal(occ.astype(bool), gh["prim"] >= 0)


def test_cornell_instanced_closest():
    print("[trace] cornell instances", flush=True)
    sc = scenes.cornell()
    ctx, arr = _ctx(sc)
    orc = native.OracleScene(arr)
    rays = np.concatenate([scenes.incoherent_rays(50000, seed=5),
                           scenes.pinhole_rays(256, 256, eye=(0.5, 0.5, -1.35), lookat=(0.5, 0.5, 0.5))])
    gh = ctx.trace_closest(rays)
    oh = orc.trace_closest(rays, tie_mode=1)
    _compare(gh, oh)
    assert set(np.unique(gh["inst"])) >= {0, 1, 2, 3, 4}


def test_tmin_tmax_window():
    print("[trace] tmin/tmax", flush=True)
    sc = scenes.soup(2000, seed=7)
    ctx, arr = _ctx(sc)
    orc = native.OracleScene(arr)
    rays = scenes.incoherent_rays(50000, seed=9)
    rng = np.random.default_rng(0)
    rays["tmin"] = rng.uniform(0, 0.3, len(rays)).astype(np.float32)
    rays["tmax"] = rng.uniform(0.3, 1.0, len(rays)).astype(np.float32)
    _compare(ctx.trace_closest(rays), orc.trace_closest(rays, tie_mode=1))
    assert np.array_equal(ctx.trace_any(rays), orc.trace_any(rays))


def test_empty_batch_and_device_entry():
    import torch
    print("[trace] empty + device", flush=True)
    sc = scenes.soup(500, seed=11)
    ctx, arr = _ctx(sc)
    assert ctx.trace_closest(np.zeros(0, lfh.RAY_DTYPE)).shape == (0,)
    rays = scenes.incoherent_rays(10000, seed=12)
    d_rays = torch.from_numpy(rays.view(np.uint8)).cuda()
    d_hits = torch.empty(len(rays) * 24, dtype=torch.uint8, device="cuda")
    ctx.trace_closest_device(d_rays.data_ptr(), len(rays), d_hits.data_ptr())
    ctx.synchronize()
    gh = d_hits.cpu().numpy().view(lfh.HIT_DTYPE)
    _compare(gh, ctx.trace_closest(rays))


def test_small_and_odd_batches_trace_every_ray():
    """Ray ids are fetched from 8 contiguous slices of the batch, each with its
    own counter: batches smaller than the slice count (slices of 0 or 1 ray)
    and sizes just around a wave's width must still trace every ray once."""
    print("[trace] small batches", flush=True)
    sc = scenes.soup(2000, seed=21)
    ctx, arr = _ctx(sc)
    orc = native.OracleScene(arr)
    rays = aimed_rays(sc, 1100, seed=22)
    for n in (1, 2, 5, 7, 8, 9, 63, 64, 65, 127, 129, 1031):
        r = np.ascontiguousarray(rays[:n])
        _compare(ctx.trace_closest(r), orc.trace_closest(r, tie_mode=1))
        assert np.array_equal(ctx.trace_any(r), orc.trace_any(r)), n


def _leaving_rays(ctx, n, seed):
    """Continuation-like rays: from the hit points of random rays, offset
    1e-3 along a new random direction (pathtrace.glsl:291), many of them
    grazing the axis-aligned walls they start on."""
    rng = np.random.default_rng(seed)
    r = scenes.incoherent_rays(n, seed=seed)
    r["org"] = rng.random((n, 3)).astype(np.float32)
    h = ctx.trace_closest(r)
    hit = h["prim"] >= 0
    p = r["org"][hit] + r["dir"][hit] * h["t"][hit][:, None]
    m = int(hit.sum())
    d = rng.normal(size=(m, 3))
    d[: m // 2, 1] *= 1e-4          # half of them nearly parallel to the floor / ceiling
    d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    out = scenes.incoherent_rays(m, seed=seed + 1)
    out["dir"] = d
    out["org"] = (p + d * 1e-3).astype(np.float32)
    return out


@pytest.mark.parametrize("device_bvh", [False, True])
def test_rays_leaving_flat_walls_match_oracle(device_bvh):
    """A ray that leaves the plane of an axis-aligned wall at distance 0 does
    not enter that wall's flat box, so it cannot hit the wall at t = -0 (the
    reference's AABBIntersect > 0 rule): the BVH4 leaves split into
    one-triangle children and the device-built tree box triangles by their
    exact vertex bounds, and hit what the reference traversal hits."""
    print(f"[trace] leaving rays device_bvh={device_bvh}", flush=True)
    sc = scenes.cornell()
    ctx = lfh.Context.from_scene(sc, device_bvh=device_bvh)
    orc = native.OracleScene(sc.arrays())
    rays = _leaving_rays(ctx, 600_000, seed=11)
    gh = ctx.trace_closest(rays)
    _compare(gh, orc.trace_closest(rays, tie_mode=1))
    assert not (gh["t"][gh["prim"] >= 0] <= 0).any()


def _hits_at_zero(v, org, d):
    """For every ray, the lowest triangle of v it hits at exactly t = 0 (-1:
    none) and whether it leaves that triangle's own box at a positive
    distance; every triangle tested, in the kernels' FP32 operations."""
    v0, e0, e1 = v[:, 0], v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]
    lo, hi = v.min(1), v.max(1)

    def cross(a, b):
        return np.stack([a[..., 1] * b[..., 2] - a[..., 2] * b[..., 1], a[..., 2] * b[..., 0] - a[..., 0] * b[..., 2],
                         a[..., 0] * b[..., 1] - a[..., 1] * b[..., 0]], -1)

    def dot(a, b):
        p = a * b
        return (p[..., 0] + p[..., 1]) + p[..., 2]

    tri = np.full(len(org), -1)
    inside = np.zeros(len(org), bool)
    with np.errstate(all="ignore"):
        for i in range(len(org)):
            pv = cross(d[i], e1)
            tv = org[i] - v0
            qv = cross(tv, e0)
            det = dot(e0, pv)
            u, w, t = dot(tv, pv) / det, dot(np.broadcast_to(d[i], qv.shape), qv) / det, dot(e1, qv) / det
            k = np.nonzero((u >= 0) & (w >= 0) & (t == 0) & (1 - u - w >= 0))[0]
            if k.size:
                tri[i] = k[0]
                inside[i] = ((np.where(d[i] > 0, hi[k[0]], lo[k[0]]) - org[i]) / d[i]).min() > 0
    return tri, inside


@pytest.mark.parametrize("device_bvh", [False, True])
def test_ties_at_distance_zero_go_to_the_lowest_triangle(device_bvh):
    """Rays that start on a mesh vertex hit every triangle around it at t = 0
    (and its copies: some triangles are there twice, the mesh in two
    instances).  The lowest (instance, prim) whose own box the ray enters (it
    leaves that box at a positive distance, the AABBIntersect > 0 rule) is in
    open boxes of every tree, so both trees must find it."""
    print(f"[trace] ties at 0 device_bvh={device_bvh}", flush=True)
    rng = np.random.default_rng(17)
    m = 33
    g = np.stack(np.meshgrid(np.arange(m), np.arange(m), indexing="ij"), -1).reshape(-1, 2) / (m - 1.0)
    p = np.concatenate([g, rng.uniform(0, 0.05, (len(g), 1))], 1)
    q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
    p = (p @ q).astype(np.float32)
    c = (np.arange(m - 1)[:, None] * m + np.arange(m - 1)).reshape(-1)
    ids = np.concatenate([np.stack([c, c + m, c + 1], 1), np.stack([c + m + 1, c + 1, c + m], 1)])
    ids = rng.permutation(ids)
    ids = np.concatenate([ids, ids[::5]])
    tris = p[ids]
    s = lfh.Scene()
    s.add_material(lfh.MATERIAL_DEFAULT)
    mesh = s.add_mesh(tris)
    s.add_instance(mesh, None, 0)
    s.add_instance(mesh, None, 0)
    s.build()
    n = 3000
    r = scenes.incoherent_rays(n, seed=19)
    r["org"] = p[rng.integers(0, len(p), n)]
    want, inside = _hits_at_zero(tris, r["org"], r["dir"])
    at0 = (want >= 0) & inside
    assert at0.sum() > 400
    ctx = lfh.Context.from_scene(s, device_bvh=device_bvh)
    got, orc = ctx.trace_closest(r), native.OracleScene(s.arrays()).trace_closest(r, tie_mode=1)
    assert np.array_equal(orc["prim"][at0], want[at0])
    bad = got["prim"][at0] != want[at0]
    assert not bad.any(), f"{bad.sum()} of {at0.sum()} rays"
    assert not got["inst"][at0].any()
    for f in ("t", "u", "v"):
        assert np.array_equal(got[f][at0].view(np.uint32), orc[f][at0].view(np.uint32)), f
    assert np.array_equal(ctx.trace_any(r).astype(bool), got["prim"] >= 0)
