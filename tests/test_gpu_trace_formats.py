"""The cone trace over FP32 and FP8 pyramids (one 16-byte texel per element; an
FP8 level is read from the decoded copy its encoder leaves), where it can go
wrong: levels smaller than a brick, images smaller than a wavefront's tile and
ragged ones, wave-uniform and per-lane cells, and a second mip chain over the
copies the first one left.

Tolerance: the trace's own, 1e-3 mean relative error against the FP32 oracle on
the downloaded pyramid (the same texels, so only the sampler's rounding
differs)."""
import numpy as np
import pytest

from gpu_util import make_app, rel_err
from oracle import binding as ob
from vct_amd import _abi as abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", [1, 2])
@pytest.mark.parametrize("aniso", [0, 1])
@pytest.mark.parametrize("warp", [0, 1])
@pytest.mark.parametrize("dim,width,height", [(16, 5, 3), (32, 67, 41)])
def test_trace_one_texel_elements(storage, aniso, warp, dim, width, height):
    app = make_app(2, dim=dim, levels=8, storage=storage, anisotropic=aniso, width=width, height=height, shadow_size=64,
                   warp_texture=warp)
    ctx, mesh = app.ctx, app.mesh()
    for frame in (0, 3):  # the second chain filters over the first one's decoded copies
        app.render(frame)
        fs, g = app.frame_state(frame), ctx.grid()
        levels = [ctx.radiance(l) for l in range(g.levels)]
        faces = [None] + [[ctx.radiance(l, f) for f in range(6)] for l in range(1, g.levels)] if aniso else None
        gbuf = ctx.download(abi.VCT_BUF_GBUFFER, 0, np.float32).reshape(height, width, 16)
        wm = np.ascontiguousarray(ctx.warp_texture()) if warp else None
        tp = ob.trace_params(fs["trace"], g.dim, g.levels, tuple(g.center), tuple(g.vmin), tuple(g.vmax),
                             mesh["rough"] is not None, aniso, wm)
        ref_i, ref_s = ob.trace(gbuf, levels, tp, aniso_faces=faces)
        ind = ctx.download(abi.VCT_BUF_INDIRECT, 0, np.float32).reshape(-1, 4)
        spec = ctx.download(abi.VCT_BUF_SPECULAR, 0, np.float32).reshape(-1, 4)
        assert rel_err(ind, ref_i) < 1e-3 and rel_err(spec, ref_s) < 1e-3, (frame, rel_err(ind, ref_i), rel_err(spec, ref_s))
    app.close()
