"""The trace's whole-tile form (images beyond the split form's sizes) over every
storage format, mip form and the warp texture: its pixels have the split form's
bits, and a part of the image agrees with the FP32 oracle on the downloaded
pyramid within the trace's own tolerance (1e-3 mean relative error; the same
texels, so only the sampler's rounding differs).  Pixels whose tangent frame is
not a number leave their neighbours alone.

A pixel's value depends on its G-buffer texel alone, so a part of the view is
traced in both forms by uploading it as an image of its own."""
import numpy as np
import pytest

from gpu_util import make_app, rel_err
from oracle import binding as ob
from vct_amd import _abi as abi

pytestmark = pytest.mark.gpu

W, H = 1100, 600  # 10,350 8x8 tiles: beyond 4096 and 8192


def _trace(ctx, cam, tr, gbuf):
    h, w = gbuf.shape[:2]
    c = abi.Camera.from_buffer_copy(cam)
    c.width, c.height = w, h
    ctx.gbuffer(c)
    ctx.upload(abi.VCT_BUF_GBUFFER, 0, np.ascontiguousarray(gbuf))
    ctx.trace(tr)
    return [ctx.download(b, 0, np.float32).reshape(h, w, 4) for b in (abi.VCT_BUF_INDIRECT, abi.VCT_BUF_SPECULAR)]


@pytest.mark.parametrize("warp", [0, 1])
@pytest.mark.parametrize("aniso", [0, 1])
@pytest.mark.parametrize("storage", [0, 1, 2])
def test_whole_tiles(storage, aniso, warp):
    app = make_app(2, dim=32, storage=storage, anisotropic=aniso, width=W, height=H, shadow_size=128,
                   warp_texture=warp)
    try:
        ctx, fs, g = app.ctx, app.frame_state(0), app.ctx.grid()
        app.render(0)
        cam, tr = fs["cam"], fs["trace"]
        assert bool(tr.warp_texture) == bool(warp) and tr.enable_reflections
        gbuf = ctx.download(abi.VCT_BUF_GBUFFER, 0, np.float32).reshape(H, W, 16)
        whole = _trace(ctx, cam, tr, gbuf)
        levels = [ctx.radiance(l) for l in range(g.levels)]
        faces = [None] + [[ctx.radiance(l, f) for f in range(6)] for l in range(1, g.levels)] if aniso else None
        wm = np.ascontiguousarray(ctx.warp_texture()) if warp else None
        tp = ob.trace_params(tr, g.dim, g.levels, tuple(g.center), tuple(g.vmin), tuple(g.vmax),
                             app.mesh()["rough"] is not None, aniso, wm)
        parts = [np.s_[0:136, 0:200], np.s_[230:366, 450:650], np.s_[464:600, 900:1100]]
        for p in parts:
            for a, b in zip(whole, _trace(ctx, cam, tr, gbuf[p])):
                assert (b != 0).any()
                assert np.array_equal(a[p].view(np.uint32), b.view(np.uint32)), p
        p = parts[1]
        for a, r in zip(whole, ob.trace(np.ascontiguousarray(gbuf[p]), levels, tp, aniso_faces=faces)):
            assert rel_err(a[p].reshape(-1, 4), r) < 1e-3, rel_err(a[p].reshape(-1, 4), r)
        # without the specular cone
        one = abi.TraceParams.from_buffer_copy(tr)
        one.enable_reflections = 0
        assert np.array_equal(_trace(ctx, cam, one, gbuf)[0].view(np.uint32), whole[0].view(np.uint32))
        # every third texel's tangent and bitangent, every fifth one's normal
        bad = gbuf.copy()
        bad[:, ::3, 8:11] = bad[:, ::3, 12:15] = np.nan
        bad[::5, 1::5, 4:7] = 0.0
        keep = np.ones((H, W), bool)
        keep[:, ::3] = keep[::5, 1::5] = False
        for a, b in zip(whole, _trace(ctx, cam, tr, bad)):
            assert np.array_equal(a[keep].view(np.uint32), b[keep].view(np.uint32))
    finally:
        app.close()


@pytest.mark.parametrize("warp", [0, 1])
@pytest.mark.parametrize("aniso", [0, 1])
def test_without_specular_cone(aniso, warp):
    """The sizes at which a launch of the diffuse cones alone changes its form:
    4096 | 4160 tiles (six directions), 8192 | 8320 (isotropic), 9216 | 9288 (six
    directions, warped)."""
    w, h = 1320, 680
    app = make_app(1, dim=32, anisotropic=aniso, width=w, height=h, shadow_size=128, warp_texture=warp, reflections=0)
    try:
        ctx, fs = app.ctx, app.frame_state(0)
        app.render(0)
        cam, tr = fs["cam"], fs["trace"]
        assert not tr.enable_reflections
        gbuf = ctx.download(abi.VCT_BUF_GBUFFER, 0, np.float32).reshape(h, w, 16)
        # every fourth column of the view beside the next ones, so that small images see surfaces
        gbuf = np.ascontiguousarray(np.concatenate([gbuf[:, k::4] for k in range(4)], 1))
        whole = _trace(ctx, cam, tr, gbuf)[0]
        assert (whole != 0).any()
        for x, y in ((512, 512), (519, 505), (1024, 512), (1032, 519), (1024, 576), (1029, 571)):
            part = _trace(ctx, cam, tr, gbuf[:y, :x])[0]
            assert np.array_equal(part.view(np.uint32), whole[:y, :x].view(np.uint32)), (x, y)
    finally:
        app.close()
