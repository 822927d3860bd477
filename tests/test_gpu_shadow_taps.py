"""The five shadow taps at the edges of a map: positions in, across and beyond
its border on every side, beyond the far plane, and positions whose
neighbouring taps' coordinates round to another texel distance than one (17
texels: s * 17 = 1/2 - 2^-25), against the oracle's composition (the tolerance
of a composed image; a tap that reads another texel changes the shadow factor
by a fifth)."""
import numpy as np
import pytest

from gpu_util import assert_compose_close, compose_variant, make_app
from oracle import binding as ob
from vct_amd import _abi as abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [16, 17, 64, 1000])
def test_shadow_taps_edges(size):
    app = make_app(1, dim=32, width=128, height=64)
    try:
        ctx, fs = app.ctx, app.frame_state(0)
        rng = np.random.default_rng(size)
        # light space = world: map coordinate s = (x + 1) / 2
        e = np.float32(1.0) / np.float32(size)
        xs = [-9.0, -1 - 9 * e, -1 - 2 * e, -1 - e, -1.0, -1 + e, 0.0, 1 - e, 1.0, 1 + e, 1 + 2 * e, 1 + 9 * e, 9.0]
        xs += [x + d for x in xs for d in (-0.3 * e, 0.45 * e, 0.7 * e)] + [986895 * 2.0 ** -24 - 1] * 8
        xs = np.asarray(xs, np.float32)
        P = np.stack([rng.choice(xs, (64, 128)), rng.choice(xs, (64, 128)), rng.uniform(-1, 1.3, (64, 128))], -1)
        g = np.zeros((64, 128, 16), np.float32)
        g[..., 0:3] = P
        g[..., 3] = np.full((64, 128), 0xffc0a080, np.uint32).view(np.float32)
        g[..., 4:8] = (0, 0, 1, 0.5)
        g[..., 8:11] = (1, 0, 0)
        g[..., 11] = np.ones((64, 128), np.uint32).view(np.float32)
        g[..., 12:15] = (0, 1, 0)
        L = abi.Light.from_buffer_copy(fs["lights"][0])
        L.type, L.enabled, L.shadow_caster, L.shadow_size, L.perspective = 1, 1, 1, size, 0
        L.direction = (0.2, -0.1, -1.0)
        L.intensity = 1.0
        L.color = (1.0, 0.9, 0.8)
        L.ls = tuple(np.eye(4, dtype=np.float32).ravel())
        L.ls_inverse = L.ls
        sm = rng.uniform(0.2, 1.0, (size, size)).astype(np.float32)
        app.build_radiance(0)
        ctx.set_lights([L])
        ctx.upload(abi.VCT_BUF_SHADOWMAP, 0, sm)
        ctx.gbuffer(fs["cam"])
        ctx.trace(fs["trace"])
        ctx.upload(abi.VCT_BUF_GBUFFER, 0, g)
        p = compose_variant(app.compose_params(0), enable_indirect=0, enable_reflections=0, enable_specular=0)
        ctx.compose(p)
        ref = ob.compose(g, None, None, [L], [sm], p)
        assert len(np.unique(np.round(ref.reshape(-1, 4)[:, 0], 4))) >= 6  # every factor occurs
        assert_compose_close(ctx.color().reshape(-1, 4), ref, f"size {size}")
    finally:
        app.close()
