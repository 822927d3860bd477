"""The injection and the mip chain over the grid sizes where their work is
split differently: rows of one to 64 bricks, runs of 1, 4 and 16 bricks per
wavefront, one region of 8^3 and fewer regions than a workgroup's wavefronts,
sources below 8^3, fp16 pairs and fp32 texels, one face and six.  Two frames of
a moving scene, so that bricks are written over an earlier frame's.  Every
texel has the oracle's bits."""
import numpy as np
import pytest

from gpu_util import make_app
from oracle import binding as ob

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("aniso", [0, 1])
@pytest.mark.parametrize("storage", [0, 1], ids=["fp16", "fp32"])
@pytest.mark.parametrize("dim", [8, 16, 64, 128, 256])
def test_level0_and_chain(dim, storage, aniso):
    app = make_app(2, dim=dim, width=64, height=64, shadow_size=256, storage=storage, anisotropic=aniso)
    try:
        ctx, g = app.ctx, app.ctx.grid()
        fp32 = storage == 1
        for frame in (0, 3):
            fs = app.frame_state(frame)
            ctx.set_transforms(fs["model"])
            ctx.shadowmaps()
            sms = [ctx.shadow(i) if L.shadow_caster else None for i, L in enumerate(fs["lights"])]
            ctx.voxelize(fs["vox"])
            alb = ctx.albedo()
            ctx.normalize_inject(fs["inj"])
            new, ref, lm, st = ob.normalize_inject(alb, g.dim, tuple(g.center), tuple(g.vmin), tuple(g.vmax),
                                                   fs["lights"], sms, fp32=fp32)
            got = ctx.radiance(0)
            assert np.array_equal(got.view(np.uint32), ref.reshape(got.shape).view(np.uint32)), frame
            assert np.array_equal(ctx.albedo(), new) and np.array_equal(ctx.litmask(), lm)
            s = ctx.stats()
            assert (s.unique_voxels, s.max_fragments_per_voxel, s.lit_voxels) == \
                (st.unique_voxels, st.max_fragments_per_voxel, st.lit_voxels)
            ctx.mip(fs["mip"])
            lv = ob.mip_aniso(got, g.levels, fp32=fp32) if aniso else ob.mip(got, g.levels, fp32=fp32)
            for l in range(1, g.levels):
                for f in range(6 if aniso else 1):
                    r = ctx.radiance(l, f)
                    want = lv[l][f] if aniso else lv[l]
                    assert np.array_equal(r.view(np.uint32), want.view(np.uint32)), (frame, l, f)
    finally:
        app.close()
