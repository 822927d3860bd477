"""The 8x8-block walk of triangles whose vertices lie up to the window clamp
(524288 px) from the image: an edge's value there passes 2^53, where FP64 has no
longer every integer.  Each triangle has a texel (named beside it) at which the
integer edge value lies within a few units of the middle between two floats, so
that a value rounded to FP64 on the way gives another barycentric.  The depth is
that barycentric (1 at its vertex, 0 at the others), and every texel has the
oracle's bits."""
import numpy as np
import pytest

from gpu_util import make_app
from oracle import binding as ob
from vct_amd import _abi as abi

pytestmark = pytest.mark.gpu

N = 2048
CASES = [  # x, y of the three vertices in NDC; the texel (column, row)
    ("0x1.e1783ep+8 -0x1.7c8e64p-10 0x1.266d6ep+1 0x1.f96ae2p+8 -0x1.8e5b9p+8 -0x1.9fe448p+8", (88, 1973)),
    ("0x1.eea9bcp+8 -0x1.b69a6cp+1 0x1.29a908p-13 0x1.f06aaap+8 -0x1.7047bap+8 -0x1.b448dep+8", (350, 233)),
    ("0x1.89ca44p+8 0x1.465aeep-3 -0x1.c156d6p+3 0x1.bd9acep+8 -0x1.969c8p+8 -0x1.8de3e6p+8", (1724, 834)),
    ("0x1.39f8p+8 0x1.353a2ep+2 -0x1.faaf3ep-9 0x1.efe31p+8 -0x1.f30866p+8 -0x1.492faap+8", (1955, 1380)),
    ("0x1.a2c68ap+8 0x1.07b89cp+1 0x1.c7b348p+0 0x1.5b1adep+8 -0x1.fd51a6p+8 -0x1.c2e358p+8", (611, 1386)),
]


def test_edge_values_beyond_2_53():
    app = make_app(1, dim=32)
    try:
        ctx = app.ctx
        eye = np.eye(4, dtype=np.float32)[None]
        L = abi.Light.from_buffer_copy(next(x for x in app.frame_state(0)["lights"] if x.shadow_caster))
        L.shadow_size, L.perspective = N, 0
        for k in range(16):
            L.ls[k] = L.ls_inverse[k] = 1.0 if k % 5 == 0 else 0.0
        ctx.set_lights([L])
        for verts, (x, y) in CASES:
            v = np.array([float.fromhex(t) for t in verts.split()], np.float32).reshape(1, 3, 2)
            z = np.array([-1, -1, 1], np.float32).reshape(1, 3, 1)
            m = {"pos": np.ascontiguousarray(np.concatenate([v, z], 2)),
                 "nrm": np.tile(np.array([0, 0, 1], np.float32), (1, 3, 1)), "tan": np.array([[1, 0, 0]], np.float32),
                 "albedo": np.full(1, 0xffffffff, np.uint32), "obj": np.zeros(1, np.uint32)}
            ctx.set_scene(m["pos"], m["nrm"], m["tan"], m["albedo"], m["obj"], 1)
            ctx.set_transforms(eye)
            ctx.shadowmaps()
            got, ref = ctx.shadow(0).view(np.uint32), ob.shadowmap(ob.SceneArrays(m, eye), L).view(np.uint32)
            assert (ref != 0x3f800000).all()  # the triangle covers the map
            assert got[y, x] == ref[y, x], (verts, x, y)
            assert np.array_equal(got, ref), verts
    finally:
        app.close()
