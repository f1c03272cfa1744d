"""The post-process kernel (postprocess.glsl) and the RGB8 read-back against
the numpy oracle (oracle/post.py) over the same accumulation: every tonemap,
chromatic aberration with and without distortion, vignette.  Float outputs
within 2e-6 relative + 1e-6 (GPU powf vs numpy); the RGB8 image equals the
oracle's conversion of the GPU's own float output.

Two places amplify float32 rounding beyond that tolerance, and the test
compares them where the rounding is not amplified:
* Uncharted 2 on black pixels computes N/D - E/F = 0 in float32 up to one ulp
  of 1/15, and x^(1/2.2) lifts 1e-8 to 2e-4.  Those cases are compared before
  the gamma, (out / (1.75 vignette))^2.2, with 5e-8 absolute.
* Chromatic aberration reads at computed texture coordinates.  A float32
  coordinate is off by up to W 2^-24 ~ 4e-6 texel, times the texel contrast at
  a light's edge, so those cases allow 1e-4 relative."""
import ctypes as C

import numpy as np
import pytest

from lavaframe_amd import lfh, scenes
from oracle import post as P

pytestmark = pytest.mark.gpu

CASES = [dict(tonemap_index=k) for k in range(7)] + [
    dict(tonemap_index=2, use_ca=1, ca_distance=0.8, ca_p2=-0.5),
    dict(tonemap_index=3, use_ca=1, use_ca_distortion=1, ca_distance=0.3, ca_p1=2.0, ca_p2=-2.0, ca_p3=0.5),
    dict(tonemap_index=1, use_vignette=1, vignette_intensity=0.9, vignette_power=1.7),
    dict(tonemap_index=6, use_ca=1, ca_distance=0.5, use_vignette=1, vignette_intensity=0.5, vignette_power=2.0),
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_post_process_matches_oracle(case):
    print(f"[post] case {case}", flush=True)
    sc = scenes.cornell(64, 48)
    ctx = lfh.Context.from_scene(sc)
    cam = sc.camera()
    ctx.update(cam, reset=True)
    ctx.render_passes(8)
    s, c = ctx.accum()
    acc = s.astype(np.float64) - c.astype(np.float64)
    pp = lfh.Postprocess.make(**CASES[case])
    inv = 1.0 / 8
    g = ctx.output_post(pp, inv)
    ref = P.postprocess(acc, inv, pp.as_dict())
    assert np.isfinite(g).all()
    rtol = 1e-4 if pp.use_ca else 2e-5
    if pp.tonemap_index == 6:
        # vignette factor per pixel: the pass over a unit image, no tonemap
        d = dict(pp.as_dict(), tonemap_index=0, use_ca=0)
        vig = P.postprocess(np.ones_like(acc), 1.0, d)
        np.testing.assert_allclose((g / (1.75 * vig)) ** 2.2, (ref / (1.75 * vig)) ** 2.2, rtol=rtol, atol=5e-8)
    else:
        np.testing.assert_allclose(g, ref, rtol=rtol, atol=2e-6)
    ldr = ctx.output_ldr(pp, inv)
    np.testing.assert_array_equal(ldr, P.to_rgb8(g))


def test_default_sample_count():
    """inv_samples <= 0 uses 1 / sample counter, like lfh_get_output_hdr."""
    sc = scenes.cornell(32, 32)
    ctx = lfh.Context.from_scene(sc)
    cam = sc.camera()
    ctx.update(cam, reset=True)
    ctx.render_passes(4)
    pp = lfh.Postprocess.make(tonemap_index=0)
    np.testing.assert_array_equal(ctx.output_post(pp), ctx.output_hdr())


@pytest.mark.parametrize("w,h", [(1, 1), (349, 251), (512, 171), (1024, 1024), (3000, 1001)])
def test_images_of_any_size_come_back_whole(w, h):
    """Images of less than a MiB, just around one, and of more MiB than the
    pinned staging holds at once (36 MB of floats): the float read-back equals
    the raw sum scaled on the host, and the RGB8 image (3 B per pixel) the
    host conversion of the post-processed floats, on a first and on a repeated
    call."""
    print(f"[post] read-back {w}x{h}", flush=True)
    sc = scenes.cornell(w, h, max_depth=2)
    ctx = lfh.Context.from_scene(sc)
    ctx.update(sc.camera(), reset=True)
    ctx.render_passes(1)
    s, c = ctx.accum()
    want = (s - c) * np.float32(1.0 / ctx.sample_count())
    for _ in range(2):
        assert np.array_equal(ctx.output_hdr().view(np.uint32), want.view(np.uint32))
    pp = lfh.Postprocess.make()
    f = ctx.output_post(pp)
    # P.to_rgb8 in the kernel's FP32: of millions of values some are within its rounding of a tie
    rgb8 = np.floor(np.clip(f, 0, 1) * np.float32(255) + np.float32(0.5)).astype(np.uint8)
    assert f.dtype == np.float32 and np.abs(rgb8.astype(int) - P.to_rgb8(f)).max() <= 1
    for _ in range(2):
        ldr = ctx.output_ldr(pp)
        assert np.array_equal(ldr, rgb8) and (w * h < 1000 or ldr.any())
    assert np.array_equal(ctx.output_hdr().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("w,h", [(64, 48), (1000, 701)])
def test_images_into_pinned_memory(w, h):
    """Images read into the caller's pinned memory equal those read into
    ordinary memory."""
    import torch
    print(f"[post] pinned {w}x{h}", flush=True)
    sc = scenes.cornell(w, h, max_depth=2)
    ctx = lfh.Context.from_scene(sc)
    ctx.update(sc.camera(), reset=True)
    ctx.render_passes(1)
    want = ctx.output_hdr()
    pin = torch.full((h, w, 3), -1.0).pin_memory()
    for _ in range(2):
        ctx._chk(ctx.lib.lfh_get_output_hdr(ctx.h, C.cast(pin.data_ptr(), lfh.f32p), w, h))
        assert np.array_equal(pin.numpy().view(np.uint32), want.view(np.uint32))
        pin.fill_(-1.0)
