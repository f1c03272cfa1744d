"""Work fetch of the persistent traversal kernels at the sizes where its rule
changes: one ray, fewer rays than waves, exactly the rays the launch's waves
own by position, one more, and a second owned round.  Every ray of a batch is
traced exactly once, so the hits of any split equal those of the CPU oracle
bit for bit (ids and the bits of t, u, v)."""
import re

import numpy as np
import pytest

from lavaframe_amd import lfh, scenes
from oracle import native

pytestmark = pytest.mark.gpu

CHUNK = int(re.search(r"#define LFH_FETCH_CHUNK (\d+)",
                      (lfh.PKG_DIR / "csrc" / "dev_trace.h").read_text()).group(1))
WAVES = 4          # per block


@pytest.fixture(scope="module")
def world():
    import torch
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    sc = scenes.soup(300, seed=3)
    # rays that one block per CU owns without dynamic fetches; a kernel's occupancy is 1 to 8 blocks
    line = cus * WAVES * CHUNK
    rays = scenes.incoherent_rays(33 * line + 77, seed=4)
    orc = native.OracleScene(sc.arrays())
    return lfh.Context.from_scene(sc), orc.trace_closest(rays), orc.trace_any(rays), rays, line


def _check(world, n):
    print(f"[fetch] {n} rays", flush=True)
    ctx, hits, occ, rays, _ = world
    r = rays[-n:]
    got, want = ctx.trace_closest(r), hits[-n:]
    for f in ("prim", "inst", "mat"):
        assert np.array_equal(got[f], want[f]), f
    for f in ("t", "u", "v"):
        assert np.array_equal(got[f].view(np.uint32), want[f].view(np.uint32)), f
    assert np.array_equal(ctx.trace_any(r), occ[-n:])


@pytest.mark.parametrize("n", [1, 7, 8, 9, 5119, 5121, 65537])
def test_every_ray_of_a_small_batch_is_traced_once(world, n):
    _check(world, n)


@pytest.mark.parametrize("blocks", range(1, 9))
@pytest.mark.parametrize("past", [-1, 0, 1])
def test_every_ray_is_traced_once_around_the_owned_share(world, blocks, past):
    """Every occupancy that a traversal kernel can have, so whatever its
    register count, one of them is the boundary of each kernel."""
    _check(world, blocks * world[4] + past)


@pytest.mark.parametrize("lines", [9, 12, 33])   # 33: a second owned round at any occupancy
def test_every_ray_of_a_large_batch_is_traced_once(world, lines):
    _check(world, lines * world[4] + 63)


@pytest.mark.parametrize("ntri", [4, 1000, 30000])
@pytest.mark.parametrize("tilt", [0.0, 1e-3])
def test_rays_through_stacked_sheets_use_the_whole_stack(ntri, tilt):
    """Parallel sheets that every ray crosses: all four children of a node are
    hit on every level, so the stack grows by three entries a level, past the
    entries kept in LDS.  Without tilt the rays are parallel to an axis (two
    infinite components of 1/d)."""
    print(f"[fetch] sheets {ntri} tilt {tilt}", flush=True)
    rng = np.random.default_rng(ntri)
    z = np.linspace(0.0, 1.0, ntri) + rng.uniform(0, 1e-6, ntri)
    v = np.zeros((ntri, 3, 3))
    v[:, 0, :2], v[:, 1, :2], v[:, 2, :2] = (-3, -3), (5, -3), (-3, 5)
    v[:, :, 2] = z[:, None]
    s = lfh.Scene()
    s.add_material(lfh.MATERIAL_DEFAULT)
    s.add_instance(s.add_mesh(v.astype(np.float32)), None, 0)
    s.build()
    n = 3000
    r = np.zeros(n, lfh.RAY_DTYPE)
    r["org"][:, :2] = rng.uniform(0.1, 0.4, (n, 2))
    # half way between sheets: a ray starting in a sheet's plane enters its flat box only
    # where the tree has grouped it with another (the distance is then 0)
    r["org"][:, 2] = (rng.integers(-ntri // 5, ntri + ntri // 5, n) + 0.5) / (ntri - 1)
    up = rng.random(n) < 0.5
    d = np.stack([np.full(n, tilt), np.full(n, 2 * tilt), np.where(up, 1.0, -1.0)], 1)
    r["dir"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    r["tmin"] = np.where(rng.random(n) < 0.3, 0.3, 0.0)     # hits behind tmin are passed over
    r["tmax"] = scenes.RAY_TMAX
    orc = native.OracleScene(s.arrays())
    want, occ = orc.trace_closest(r), orc.trace_any(r)
    for device_bvh in (False, True):
        ctx = lfh.Context.from_scene(s, device_bvh=device_bvh)
        got = ctx.trace_closest(r)
        for f in ("prim", "inst"):
            assert np.array_equal(got[f], want[f]), (f, device_bvh)
        for f in ("t", "u", "v"):
            assert np.array_equal(got[f].view(np.uint32), want[f].view(np.uint32)), (f, device_bvh)
        assert np.array_equal(ctx.trace_any(r), occ), device_bvh
        ctx.close()
