"""The trace's two work splits at the sizes where a launch changes from one to
the other and at their edges: one pixel, less than a tile, ragged tiles, tiles
whose right or bottom part is outside the image, the last size of the split
form and the first of the other, with and without the specular cone.

The cones are traced and added by the same code in the same order, so a
picture's top left part has the same bits whatever the image size: the view of
a camera is sampled through an uploaded G-buffer whose texels do not depend on
the image's size."""
import numpy as np
import pytest

from gpu_util import make_app, rel_err
from oracle import binding as ob
from vct_amd import _abi as abi

pytestmark = pytest.mark.gpu


def _trace(ctx, cam, tr, gbuf, w, h):
    c = abi.Camera.from_buffer_copy(cam)
    c.width, c.height = w, h
    ctx.gbuffer(c)
    ctx.upload(abi.VCT_BUF_GBUFFER, 0, np.ascontiguousarray(gbuf[:h, :w]))
    ctx.trace(tr)
    ind = ctx.download(abi.VCT_BUF_INDIRECT, 0, np.float32).reshape(h, w, 4)
    spec = ctx.download(abi.VCT_BUF_SPECULAR, 0, np.float32).reshape(h, w, 4)
    return ind.view(np.uint32), spec.view(np.uint32)


# 8x8 tiles: 512 | 513 (six parts), 4096 | 4160 (six directions), 8192 | 8320 (isotropic)
SIZES = [(1, 1), (7, 9), (65, 3), (256, 128), (257, 127), (512, 512), (519, 505), (1024, 512), (1032, 519)]


@pytest.mark.parametrize("refl", [0, 1])
@pytest.mark.parametrize("aniso", [0, 1])
def test_split_and_whole_tiles_agree(aniso, refl):
    app = make_app(1, dim=32, anisotropic=aniso, width=1100, height=600, reflections=refl)
    ctx, fs = app.ctx, app.frame_state(0)
    app.build_radiance(0)
    cam, tr = fs["cam"], fs["trace"]
    ctx.gbuffer(cam)
    gbuf = ctx.download(abi.VCT_BUF_GBUFFER, 0, np.float32).reshape(600, 1100, 16)
    # a busy corner: every third column of the view, so that small images see
    # surfaces and some of their texels are uncovered
    gbuf = np.ascontiguousarray(np.concatenate([gbuf[:, ::3], gbuf[:, 1::3], gbuf[:, 2::3]], 1))
    gbuf[::5, ::7] = 0
    whole_i, whole_s = _trace(ctx, cam, tr, gbuf, 1100, 600)
    assert (whole_i != 0).any()
    for w, h in SIZES:
        ind, spec = _trace(ctx, cam, tr, gbuf, w, h)
        assert np.array_equal(ind, whole_i[:h, :w]), (w, h)
        if refl:
            assert np.array_equal(spec, whole_s[:h, :w]), (w, h)
    # and the small form against the oracle (the trace's tolerance)
    g = ctx.grid()
    levels = [ctx.radiance(l) for l in range(g.levels)]
    faces = [None] + [[ctx.radiance(l, f) for f in range(6)] for l in range(1, g.levels)] if aniso else None
    ind, spec = _trace(ctx, cam, tr, gbuf, 65, 63)
    tp = ob.trace_params(tr, g.dim, g.levels, tuple(g.center), tuple(g.vmin), tuple(g.vmax),
                         app.mesh()["rough"] is not None, aniso)
    ref_i, ref_s = ob.trace(np.ascontiguousarray(gbuf[:63, :65]), levels, tp, aniso_faces=faces)
    assert rel_err(ind.view(np.float32).reshape(-1, 4), ref_i) < 1e-3
    if refl:
        assert rel_err(spec.view(np.float32).reshape(-1, 4), ref_s) < 1e-3
    app.close()
