"""The 8x8-block walk of large triangles at its edges: images that blocks
overhang, images below one block, one-pixel rows, triangles that span runs of
blocks (so that runs enter them mid-way), 32-bit and FP64 edge values (the
latter for boxes past the small form's 4096 px), equal depths, and more
fragments per pixel than a wavefront's.  Every texel has the oracle's bits."""
import numpy as np
import pytest

from gpu_util import make_app
from oracle import binding as ob
from vct_amd import _abi as abi

pytestmark = pytest.mark.gpu


def _soup(base, n, seed):
    """n triangles from slivers to several times the scene's extent, a quarter
    of them drawn twice (equal depths), around the scene's own box."""
    rng = np.random.default_rng(seed)
    lo, hi = base.reshape(-1, 3).min(0), base.reshape(-1, 3).max(0)
    c = rng.uniform(lo, hi, (n, 1, 3))
    size = (hi - lo).max() * 2.0 ** rng.uniform(-7, 1.5, (n, 1, 1))
    pos = (c + rng.standard_normal((n, 3, 3)) * size).astype(np.float32)
    pos[n - n // 4:] = pos[:n // 4]
    nrm = np.cross(pos[:, 1] - pos[:, 0], pos[:, 2] - pos[:, 0])
    nrm = (nrm / np.linalg.norm(nrm, axis=1, keepdims=True)).astype(np.float32)
    tan = (pos[:, 1] - pos[:, 0]).astype(np.float32)
    return {"pos": pos, "nrm": np.repeat(nrm[:, None], 3, 1), "tan": tan,
            "albedo": rng.integers(0, 2 ** 32, n, dtype=np.uint32), "obj": np.zeros(n, np.uint32)}


@pytest.mark.parametrize("n", [1, 37, 400])
def test_block_walk_edges(n):
    app = make_app(1, dim=32)
    try:
        ctx, fs = app.ctx, app.frame_state(0)
        mesh = app.mesh()
        eye = np.eye(4, dtype=np.float32)[None]
        m = _soup(mesh["pos"], n, n)
        ctx.set_scene(m["pos"], m["nrm"], m["tan"], m["albedo"], m["obj"], 1)
        ctx.set_transforms(eye)
        sc = ob.SceneArrays(m, eye)
        base = next(L for L in fs["lights"] if L.shadow_caster)
        lights = []
        for size in (16, 17, 200, 1000, 2055, 4500):
            L = abi.Light.from_buffer_copy(base)
            L.shadow_size = size
            lights.append(L)
        ctx.set_lights(lights)
        ctx.shadowmaps()
        for i, L in enumerate(lights):
            ref = ob.shadowmap(sc, L)
            assert np.array_equal(ctx.shadow(i).view(np.uint32), ref.view(np.uint32)), (n, L.shadow_size)
            assert n == 1 or (ref < 1.0).any()
        for w, h in ((1, 1), (9, 7), (1000, 1), (131, 200), (1921, 67), (4500, 40)):
            cam = abi.Camera.from_buffer_copy(fs["cam"])
            cam.width, cam.height = w, h
            ctx.gbuffer(cam)
            got = ctx.download(abi.VCT_BUF_GBUFFER, 0, np.float32).reshape(h, w, 16)
            assert np.array_equal(got.view(np.uint32), ob.gbuffer(sc, cam).view(np.uint32)), (n, w, h)
    finally:
        app.close()


@pytest.mark.parametrize("n", [2047, 2048, 2049, 16384, 16385])
def test_slot_counts(n):
    """Item offsets at the edges of a tile of slots and of the count up to
    which a tile adds up the slots in front of it itself, small triangles and
    a few that cover the whole map (more chunks of items than slots)."""
    app = make_app(1, dim=32)
    try:
        ctx, fs = app.ctx, app.frame_state(0)
        eye = np.eye(4, dtype=np.float32)[None]
        m = _soup(app.mesh()["pos"], n, n)
        c = m["pos"].mean(1, keepdims=True)
        keep = np.random.default_rng(1).random((n, 1, 1)) < 0.995
        m["pos"] = np.where(keep, c + (m["pos"] - c) * np.float32(0.02), m["pos"]).astype(np.float32)
        ctx.set_scene(m["pos"], m["nrm"], m["tan"], m["albedo"], m["obj"], 1)
        ctx.set_transforms(eye)
        sc = ob.SceneArrays(m, eye)
        L = abi.Light.from_buffer_copy(next(L for L in fs["lights"] if L.shadow_caster))
        L.shadow_size = 200
        ctx.set_lights([L])
        ctx.shadowmaps()
        ref = ob.shadowmap(sc, L)
        assert (ref < 1.0).any()
        assert np.array_equal(ctx.shadow(0).view(np.uint32), ref.view(np.uint32))
        ctx.voxelize(fs["vox"])
        alb, nrm, st = ob.voxelize(sc, [L], [ref], fs["vox"], 32)
        assert np.array_equal(ctx.albedo(), alb) and np.array_equal(ctx.normal(), nrm)
        assert ctx.stats().total_voxel_fragments == st.total_voxel_fragments
    finally:
        app.close()


@pytest.mark.parametrize("n", [70, 2000, 2500, 9000])
def test_sparse_slots(n):
    """Chunks of items whose slots lie far apart: all but a few triangles are
    too small to cover anything, so that a chunk spans from under 64 to
    thousands of slots; items of both passes, samples and statistics."""
    app = make_app(1, dim=64)
    try:
        ctx, fs = app.ctx, app.frame_state(0)
        eye = np.eye(4, dtype=np.float32)[None]
        m = _soup(app.mesh()["pos"], n, n)
        c = m["pos"].mean(1, keepdims=True)
        scale = np.full((n, 1, 1), 1e-6, np.float32)
        scale[:: max(1, n // 12)] = 0.05  # a dozen of a few pixels each
        scale[n // 2:: max(1, n // 3)] = 1.0
        m["pos"] = (c + (m["pos"] - c) * scale).astype(np.float32)
        ctx.set_scene(m["pos"], m["nrm"], m["tan"], m["albedo"], m["obj"], 1)
        ctx.set_transforms(eye)
        sc = ob.SceneArrays(m, eye)
        L = abi.Light.from_buffer_copy(next(L for L in fs["lights"] if L.shadow_caster))
        L.shadow_size = 256
        ctx.set_lights([L])
        ctx.shadowmaps()
        ref = ob.shadowmap(sc, L)
        assert np.array_equal(ctx.shadow(0).view(np.uint32), ref.view(np.uint32))
        ctx.voxelize(fs["vox"])
        alb, nrm, st = ob.voxelize(sc, [L], [ref], fs["vox"], 64)
        assert (alb != 0).any()
        assert np.array_equal(ctx.albedo(), alb) and np.array_equal(ctx.normal(), nrm)
        assert ctx.stats().total_voxel_fragments == st.total_voxel_fragments
    finally:
        app.close()
