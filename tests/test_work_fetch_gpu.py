"""Work fetch of the persistent traversal kernels at the sizes where its rule
changes: one ray, fewer rays than waves, exactly the rays the launch's waves
own by position, one more, and a second owned round.  Every ray of a batch is
traced exactly once, so the hits of any split equal those of the CPU oracle
bit for bit (ids and the bits of t, u, v)."""
import numpy as np
import pytest

from lavaframe_amd import lfh, scenes
from oracle import native

pytestmark = pytest.mark.gpu

# 256 CUs x 5 or 6 blocks x 4 waves x 64 rays: the largest queues without dynamic fetches
CLOSEST, ANY = 256 * 5 * 4 * 64, 256 * 6 * 4 * 64


@pytest.fixture(scope="module")
def world():
    sc = scenes.soup(300, seed=3)
    rays = scenes.incoherent_rays(4 * ANY + 77, seed=4)
    return lfh.Context.from_scene(sc), native.OracleScene(sc.arrays()), rays


@pytest.mark.parametrize("n", [1, 7, 8, 9, 5119, 5121, 65537, CLOSEST - 1, CLOSEST, CLOSEST + 1, ANY - 1, ANY + 1,
                               2 * CLOSEST + 63, 4 * ANY + 77])
def test_every_ray_of_a_batch_is_traced_once(world, n):
    print(f"[fetch] {n} rays", flush=True)
    ctx, orc, rays = world
    r = rays[-n:]
    got, want = ctx.trace_closest(r), orc.trace_closest(r)
    for f in ("prim", "inst", "mat"):
        assert np.array_equal(got[f], want[f]), f
    for f in ("t", "u", "v"):
        assert np.array_equal(got[f].view(np.uint32), want[f].view(np.uint32)), f
    assert np.array_equal(ctx.trace_any(r), orc.trace_any(r))
