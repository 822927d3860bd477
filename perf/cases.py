"""The work a program has this framework do, as cases that can be timed.

Kinds of case:
  frame   App.render: every pass of a frame (shadow maps, voxelize, inject,
          mip, G-buffer, cone trace, composition), from the smallest preview to
          the warped 4K scene, over the storage formats and the app's options.
  volume  App.build_radiance: the lighting volume alone, for a program that
          updates it without drawing.
  gather  vct_trace alone: another view of a volume that did not change.
  mip     vct_mip alone: both chains of an injected volume.
  train   vct_learned_train: the learned gather's network, trained from scratch.
  infer   vct_trace_learned: its image.
  labels  vct_learned_prepare: labels and features of new training points.

The frames are the generated scenes of the application layer (1: a room and two
boxes, 2: 351,680 triangles in 2,064 moving objects, 5: scene 2's distributions
with 2,717,440 triangles), seeded.  A frame's results stay on the GPU, where
the next pass and the next frame use them: run() returns them as a view that
reads a buffer back when it is looked at (the `read` frames return the picture
itself, as a program that saves it does).
"""
from __future__ import annotations

import math

import numpy as np
import torch

import vct_amd
from vct_amd import _abi as abi

FP16, FP32, FP8 = 0, 1, 2
ROOM, OBJECTS, LARGE = 1, 2, 5
TRIANGLES = {ROOM: 36, OBJECTS: 351_680, LARGE: 2_717_440}
LIGHTS = {ROOM: 1, OBJECTS: 5, LARGE: 8}


def _case(kind, name=None, **kw):
    base = dict(kind=kind, scene=OBJECTS, dim=256, storage=FP16, aniso=True, width=256, height=256, shadow=1024)
    if kind == "frame":
        base.update(frames=2, read=False, msaa=True, lighting=True, reflections=True, fill=False, tess=False, warp=False)
    base.update(kw)
    if name is not None:
        base["name"] = name
    return base


def listed():
    return [
        # a thumbnail or an interactive edit of a small room, read back each time: launches and latency
        _case("frame", "preview", scene=ROOM, dim=64, aniso=False, shadow=512, reflections=False, frames=1, read=True),
        # the static room at a common window size, the reference's own mip chain (isotropic)
        _case("frame", "room_720p", scene=ROOM, dim=128, aniso=False, shadow=1024, width=1280, height=720),
        # the moving scene the repository's benchmark quotes: 256^3, six-direction mips, 1080p
        _case("frame", "objects_1080p", width=1920, height=1080),
        # the largest configuration: 2.7M triangles, 8 lights, warp texture, FP8 coarse levels, 4K
        _case("frame", "large_4k", scene=LARGE, storage=FP8, warp=True, width=3840, height=2160, frames=1),
        # an odd window, full-precision storage, single-sample voxels, holes filled, a larger main shadow map
        _case("frame", "objects_fp32_odd", dim=128, storage=FP32, aniso=False, width=1279, height=719, shadow=2048,
              msaa=False, fill=True),
        # the tessellation voxelizer and FP8 storage in a small odd window
        _case("frame", "objects_tess", dim=128, storage=FP8, width=961, height=541, tess=True),
        # the largest grid: only the volume is rebuilt
        _case("volume", "volume_512", dim=512, aniso=False),
        # a new view of a standing volume: six-direction fp16, and isotropic fp32 in an odd window
        _case("gather", "gather_aniso", width=1280, height=720),
        _case("gather", "gather_fp32", scene=ROOM, dim=64, storage=FP32, aniso=False, width=1001, height=567),
        # training the learned gather (the configured batch), and drawing with it at 1080p
        _case("train", "train", scene=ROOM, dim=64, aniso=False, batch=4096, steps=128, points=65536),
        _case("infer", "infer_1080p", scene=ROOM, dim=64, aniso=False, width=1920, height=1080),
        # labels and features of a set of new training points
        _case("labels", "labels", scene=ROOM, dim=64, aniso=False, points=32768),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "volume", "gather", "gather", "mip", "train", "infer", "labels"])
    scene = rng.choice([ROOM, OBJECTS])
    storage = rng.choice([FP16, FP16, FP32, FP8])
    aniso = rng.random() < 0.5
    size = dict(width=_log(rng, 90, 1920), height=_log(rng, 70, 1080), shadow=_log(rng, 200, 2048))
    dim = rng.choice([32, 64, 128, 256])
    if kind == "frame":
        return _case(kind, scene=scene, dim=dim, storage=storage, aniso=aniso, frames=rng.choice([1, 2]),
                     read=rng.random() < 0.2, msaa=rng.random() < 0.8, lighting=rng.random() < 0.8,
                     reflections=rng.random() < 0.7, fill=rng.random() < 0.2, tess=rng.random() < 0.2,
                     warp=rng.random() < 0.2, **size)
    if kind == "volume":
        return _case(kind, scene=scene, dim=rng.choice([32, 64, 128, 256, 512]), storage=rng.choice([FP16, FP8]),
                     aniso=False, shadow=size["shadow"])
    if kind == "gather":
        size["width"], size["height"] = min(size["width"], 1400), min(size["height"], 800)
        return _case(kind, scene=scene, dim=dim, storage=storage, aniso=aniso, **size)
    if kind == "mip":
        return _case(kind, scene=scene, dim=dim, storage=storage, aniso=aniso, shadow=size["shadow"])
    dim = rng.choice([32, 64, 128])
    if kind == "train":
        return _case(kind, scene=ROOM, dim=dim, storage=storage, aniso=False, batch=64 * _log(rng, 1, 128),
                     steps=_log(rng, 8, 128), points=_log(rng, 1000, 100_000))
    if kind == "infer":
        return _case(kind, scene=ROOM, dim=dim, storage=storage, aniso=False, **size)
    return _case(kind, scene=ROOM, dim=dim, storage=storage, aniso=False, points=_log(rng, 500, 32768))


# --- the program ------------------------------------------------------------------
def _app(case, seed):
    fr = case["kind"] == "frame"
    app = vct_amd.App(case["scene"], seed=1 + seed % 1_000_003, dim=case["dim"], storage=case["storage"],
                      anisotropic=int(case["aniso"]), width=case["width"], height=case["height"],
                      shadow_size=case["shadow"], reflections=int(case["reflections"]) if fr else 1,
                      msaa=int(case["msaa"]) if fr else 1, lighting=int(case["lighting"]) if fr else 1,
                      fill_holes=int(case["fill"]) if fr else 0, tessellation=int(case["tess"]) if fr else 0,
                      warp_texture=int(case["warp"]) if fr else 0)
    app.ctx.set_timing(False)  # the pass timers are for profiling
    return app


def prepare(case, seed):
    app = _app(case, seed)
    ctx, kind = app.ctx, case["kind"]
    st = {"case": case, "app": app, "ctx": ctx, "first": seed % 61}
    if kind in ("frame", "volume"):
        return st
    app.build_radiance(st["first"])
    fs = app.frame_state(st["first"])
    st["trace"], st["mip"] = fs["trace"], fs["mip"]
    if kind in ("gather", "infer"):
        ctx.gbuffer(app.camera(seed))
    if kind in ("train", "labels"):
        ctx.learned_set_points(app.surface_points(case["points"], st["first"], seed=1 + seed))
    if kind == "infer":
        ctx.learned_set_points(app.surface_points(16384, st["first"], seed=1 + seed))
        ctx.learned_prepare()
        ctx.learned_train(steps=200, batch=2048, lr=1e-3, seed=1 + seed % 1000, reset=True)
    if kind == "train":
        ctx.learned_prepare()
        st["seed"] = 1 + seed % 1000
    return st


class Buffers(dict):
    """What a pass left in the context's buffers: each one is read back when it is looked at."""

    def __init__(self, ctx, names):
        super().__init__((n, None) for n in names)
        self.ctx = ctx

    def __getitem__(self, name):
        what, _, at = name.partition(" ")
        c = self.ctx
        if what == "radiance":
            level, face = (int(v) for v in at.split("."))
            return c.radiance(level, face)
        if what in ("albedo", "normal"):
            return c.download(abi.VCT_BUF_ALBEDO if what == "albedo" else abi.VCT_BUF_NORMAL, int(at or 0), np.int32)
        if what == "shadow":
            return c.shadow(int(at))
        if what == "features":
            return torch.from_numpy(c.download(abi.VCT_BUF_FEATURES, 0, np.int16)).view(torch.bfloat16)
        if what == "stats":
            s = c.stats()
            return [int(s.total_voxel_fragments), int(s.unique_voxels), int(s.max_fragments_per_voxel), int(s.lit_voxels)]
        buf = {"color": abi.VCT_BUF_COLOR, "indirect": abi.VCT_BUF_INDIRECT, "specular": abi.VCT_BUF_SPECULAR,
               "labels": abi.VCT_BUF_LABELS}[what]
        return c.download(buf, 0, np.float32).reshape(-1, 4)

    def items(self):
        return [(n, self[n]) for n in self]

    def values(self):
        return [self[n] for n in self]


def _levels(ctx, first=0):
    """The names of the radiance volumes of levels first .. the last."""
    g = ctx.grid()
    return ["radiance %d.%d" % (l, f) for l in range(first, g.levels) for f in range(6 if g.anisotropic and l else 1)]


def run(st):
    case, app, ctx = st["case"], st["app"], st["ctx"]
    kind = case["kind"]
    if kind == "frame":
        for k in range(case["frames"]):
            app.render(st["first"] + k)
        if case["read"]:
            return {"color": ctx.color()}
        names = ["color", "indirect", "albedo", "normal", "stats"] + (["specular"] if case["reflections"] else [])
        return Buffers(ctx, names + ["shadow %d" % i for i in range(LIGHTS[case["scene"]])] + _levels(ctx))
    if kind == "volume":
        app.build_radiance(st["first"])
        return Buffers(ctx, ["albedo", "normal", "stats"] + ["shadow %d" % i for i in range(LIGHTS[case["scene"]])] + _levels(ctx))
    if kind == "gather":
        ctx.trace(st["trace"])
        return Buffers(ctx, ["indirect", "specular"])
    if kind == "mip":
        ctx.mip(st["mip"])
        return Buffers(ctx, ["albedo %d" % l for l in range(1, ctx.grid().levels)] + _levels(ctx, 1))
    if kind == "train":
        loss = ctx.learned_train(steps=case["steps"], batch=case["batch"], lr=1e-3, seed=st["seed"], reset=True)
        return {"loss": loss, "weights": ctx.weights()}
    if kind == "infer":
        ctx.trace_learned(st["trace"], math.inf, count_fallback=False)
        return Buffers(ctx, ["indirect"])
    ctx.learned_prepare()
    return Buffers(ctx, ["labels", "features"])


# --- what a pass cannot do without ----------------------------------------------------
MLP_MACS = 129 * 64 + 64 * 64 + 64 * 64 + 64 * 3


def work(case):
    kind, dim, px = case["kind"], case["dim"], case["width"] * case["height"]
    nv, texel = dim ** 3, 16 if case["storage"] == FP32 else 8
    upper = sum(max(1, dim >> l) ** 3 for l in range(1, int(math.log2(dim)) + 1)) * (6 if case["aniso"] else 1)
    tri, nl, sm = TRIANGLES[case["scene"]], LIGHTS[case["scene"]], case["shadow"] ** 2
    shadow = nl * (tri * 40 + sm * 4)
    volume = tri * 80 + 8 * nv + 4 * nv + nl * sm * 4 + nv * texel + (nv + upper) * texel + 4 * nv * 9 / 8
    image = px * (64 + 32) + (nv + upper) * texel  # a G-buffer texel read, two image texels written, the pyramid once
    # about eight samples a cone, each two levels of eight corners of four channels (three faces if directional)
    gather = px * 7 * 8 * 2 * 8 * 4 * 2 * (3 if case["aniso"] else 1)
    if kind == "frame":
        draw_px = tri * 80 + px * (64 + 64 + 32 + 16 + 16)
        n = case["frames"]
        return {"bytes": n * (shadow + volume + draw_px + (nv + upper) * texel), "flops": n * gather}
    if kind == "volume":
        return {"bytes": shadow + volume, "flops": 0}
    if kind == "gather":
        return {"bytes": image, "flops": gather}
    if kind == "mip":
        return {"bytes": (nv + upper) * texel + 4 * nv * 9 / 8, "flops": 0}
    if kind == "train":
        rows = case["batch"] * case["steps"]
        return {"bytes": rows * (160 * 2 + 16) + case["steps"] * 16835 * 4 * 6, "flops": rows * 2 * (3 * MLP_MACS - 129 * 64)}
    if kind == "infer":
        return {"bytes": px * (64 + 16) + (dim // 4) ** 3 * texel, "flops": px * 2 * MLP_MACS}
    # labels: 64 cones of about 40 samples each
    return {"bytes": case["points"] * (64 + 16 + 320) + (nv + upper) * texel, "flops": case["points"] * 64 * 40 * 2 * 8 * 4 * 2}


# --- the same results in 64 bits, from the same inputs ------------------------------------
# The inputs of a pass (the stored pyramid, the G-buffer, the points, the first
# weights) are read from a prepared state; what the pass computes from them is
# plain torch in float64.  Whole frames and volumes have none: they begin with
# the rasterization of up to millions of triangles.
CONES = [((0.0, 1.0, 0.0), 0.25), ((0.0, 0.5, 0.866025), 0.15), ((0.823639, 0.5, 0.267617), 0.15),
         ((0.509037, 0.5, -0.700629), 0.15), ((-0.5909037, 0.5, -0.700629), 0.15), ((-0.823639, 0.5, 0.267617), 0.15)]


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _pyramid(ctx):
    """Every level as [faces, s, s, s, 4] float32 (the stored values)."""
    g = ctx.grid()
    out = []
    for l in range(g.levels):
        nf = 6 if g.anisotropic and l else 1
        out.append(torch.stack([torch.from_numpy(ctx.radiance(l, f)) for f in range(nf)]).to(_dev()))
    return out


def _linear(vol, p, d=None):
    """GL LINEAR of a level at p [n, 3] in [0, 1], border 0; with six faces, the
    d^2-weighted mix of the three that face the directions d."""
    nf, s = vol.shape[0], vol.shape[1]
    flat = vol.reshape(-1, 4)
    u = p * s - 0.5
    i0 = torch.floor(u).long()
    f = u - i0
    out = torch.zeros(p.shape[0], 4, dtype=torch.float64, device=p.device)
    for c in range(8):
        o = torch.tensor([c & 1, (c >> 1) & 1, c >> 2], device=p.device)
        i = i0 + o
        w = torch.where(o.bool(), f, 1 - f).prod(1) * ((i >= 0) & (i < s)).all(1)
        i = i.clamp(0, s - 1)
        e = (i[:, 2] * s + i[:, 1]) * s + i[:, 0]
        if nf == 1:
            out += w[:, None] * flat[e].double()
        else:
            for a in range(3):
                face = 2 * a + (d[:, a] < 0).long()
                out += (w * d[:, a] ** 2)[:, None] * flat[face * s ** 3 + e].double()
    return out


def _mipmapped(levels, p, lam, d=None):
    """LINEAR_MIPMAP_LINEAR at the level lam (one number), NEAREST of level 0 where lam <= 0."""
    q = len(levels) - 1
    if lam <= 0:
        s = levels[0].shape[1]
        i = torch.floor(p * s).long()
        ok = ((i >= 0) & (i < s)).all(1)
        i = i.clamp(0, s - 1)
        return levels[0][0][i[:, 2], i[:, 1], i[:, 0]].double() * ok[:, None]
    if lam >= q:
        return _linear(levels[q], p, d)
    l = min(int(math.floor(lam)), q - 1)
    fr = lam - l
    return (1 - fr) * _linear(levels[l], p, d) + fr * _linear(levels[l + 1], p, d)


def _cone(levels, start, d, steps, tan_half, h, offset, dim, stop, label=False):
    """March of cones from `start` along the unit directions d: [n, 4]."""
    acc = torch.zeros(start.shape[0], 4, dtype=torch.float64, device=start.device)
    live = torch.arange(start.shape[0], device=start.device)
    for _ in range(steps):
        p = start[live] + h * d[live] / dim
        ok = ((p >= 0) & (p <= 1)).all(1) & (acc[live, 3] < stop)
        live, p = live[ok], p[ok]
        if not len(live):
            break
        r = h * tan_half
        s = _mipmapped(levels, p, math.log2(max(1.0, 2 * r)) + offset, d[live])
        if label:  # quarter-diameter steps: half the radiance, the opacity of half the length
            s = torch.cat([0.5 * s[:, :3], 1 - torch.sqrt(1 - s[:, 3:].clamp(0, 1))], 1)
        acc[live] += (1 - acc[live, 3:]) * s
        h += (0.5 if label else 1.0) * r
    return acc


def _unit(v):
    return v / v.norm(dim=1, keepdim=True)


def _texels(ctx, g):
    """Position in [0, 1], normal, tangent and bitangent of covered G-buffer texels g [n, 16]."""
    gd = ctx.grid()
    lo, hi, mid = (torch.tensor(list(v), dtype=torch.float64, device=g.device) for v in (gd.vmin, gd.vmax, gd.center))
    x = g.double()
    return (x[:, 0:3] - mid - lo) / (hi - lo), x[:, 4:7], x[:, 8:11], x[:, 12:15]


def _gbuffer(ctx):
    g = torch.from_numpy(ctx.download(abi.VCT_BUF_GBUFFER, 0, np.float32).reshape(-1, 16)).to(_dev())
    return g, (g[:, 11].contiguous().view(torch.int32) != 0).nonzero()[:, 0]


def _exact_gather(st):
    ctx, tr = st["ctx"], st["trace"]
    levels = _pyramid(ctx)
    g, cov = _gbuffer(ctx)
    dim = ctx.grid().dim
    ind = torch.zeros(g.shape[0], 4, dtype=torch.float64, device=g.device)
    spec = ind.clone()
    eye = torch.tensor(list(tr.eye), dtype=torch.float64, device=g.device)
    rough = tr.cone_angle_from_roughness and st["app"].mesh()["rough"] is not None
    for at in cov.split(1 << 18):
        pos, n, t, b = _texels(ctx, g[at])
        unit = _unit(n)
        D = tr.diffuse
        total = torch.zeros(len(at), 4, dtype=torch.float64, device=g.device)
        for c, w in CONES:
            d = _unit(t * c[0] + b * c[1] + n * c[2])
            total += w * _cone(levels, pos + D.bias * unit / dim, d, D.steps, math.tan(D.cone_angle / 2),
                               D.cone_initial_height, D.lod_offset, dim, 0.95)
        occ = 1 - total[:, 3:].clamp(0, 1)
        ind[at] = torch.cat([total[:, :3] * (occ if tr.draw_occlusion else 1.0), occ], 1)
        S = tr.specular
        i = g[at, 0:3].double() - eye
        r = _unit(i - 2 * (unit * i).sum(1, keepdim=True) * unit)
        angles = (g[at, 7].double() * 3.1415982 * 0.1) if rough else torch.full_like(r[:, 0], S.cone_angle)
        part = torch.zeros_like(total)
        for a in angles.unique().tolist():
            k = (angles == a).nonzero()[:, 0]
            part[k] = _cone(levels, pos[k] + S.bias * unit[k] / dim, r[k], S.steps, math.tan(a / 2),
                            S.cone_initial_height, S.lod_offset, dim, 0.95)
        spec[at] = part
    return {"indirect": ind.cpu(), "specular": spec.cpu() if tr.enable_reflections else None}


def _exact_mip(st):
    ctx = st["ctx"]
    g = ctx.grid()
    vols = [torch.from_numpy(ctx.radiance(0)).to(_dev()).double()] * (6 if g.anisotropic else 1)
    out = {}
    for l in range(1, g.levels):
        for f, v in enumerate(vols):
            s = v.shape[0] // 2
            c = v.reshape(s, 2, s, 2, s, 2, 4)
            if g.anisotropic:  # front-to-back pairs along the face's axis, the mean of the four
                a, neg = f >> 1, f & 1
                dim = {0: 5, 1: 3, 2: 1}[a]
                near, far = c.select(dim, neg), c.select(dim, 1 - neg)
                near = near + (1 - near[..., 3:]) * far
                c = near.mean([k for k, at in enumerate([0, 1, 2, 3, 4, 5, 6][:dim] + [0, 1, 2, 3, 4, 5, 6][dim + 1:])
                               if at in (1, 3, 5)])
            else:
                c = c.mean([1, 3, 5])
            out["radiance %d.%d" % (l, f)] = c.cpu()
            vols = vols[:f] + [c] + vols[f + 1:]
    return out


def _features(ctx, g):
    """The 129 inputs of the network for covered texels g [n, 16]."""
    pos, _, _, b = _texels(ctx, g)
    level = torch.from_numpy(ctx.radiance(2)).to(g.device)[None]
    s = level.shape[1]
    cols = []
    for z in (-1, 0, 1):
        for y in (-1, 0, 1):
            for x in (-1, 0, 1):
                o = torch.tensor([x, y, z], dtype=torch.float64, device=g.device) / s
                cols.append(_linear(level, pos + o))
    cols.append(_unit(b))
    for c in range(3):
        for f in (1, 2, 4):
            a = math.pi * f * pos[:, c]
            cols += [torch.sin(a)[:, None], torch.cos(a)[:, None]]
    return torch.cat(cols, 1)


def _points(st, seed):
    c = st["case"]
    return torch.from_numpy(st["app"].surface_points(c["points"], st["first"], seed=1 + seed)).to(_dev())


def _exact_labels(st, seed):
    ctx, pts = st["ctx"], _points(st, seed)
    levels, dim = _pyramid(ctx), ctx.grid().dim
    golden = math.pi * (3 - math.sqrt(5))
    out = []
    for g in pts.split(4096):
        pos, n, t, b = _texels(ctx, g)
        start = pos + _unit(n) / dim
        total = torch.zeros(g.shape[0], 4, dtype=torch.float64, device=g.device)
        for i0 in range(0, 64, 16):
            ds, ws = [], []
            for i in range(i0, i0 + 16):
                y = 1 - (i + 0.5) / 64
                r = math.sqrt(1 - y * y)
                ds.append(_unit(t * (r * math.cos(golden * i)) + b * y + n * (r * math.sin(golden * i))))
                ws.append(y / 32)
            c = _cone(levels, start.repeat(16, 1), torch.cat(ds), 256, math.tan(math.radians(10)), 1.0, 0.5, dim, 0.999, True)
            total += (c.reshape(16, -1, 4) * torch.tensor(ws, dtype=torch.float64, device=g.device)[:, None, None]).sum(0)
        occ = 1 - total[:, 3:].clamp(0, 1)
        out.append(torch.cat([total[:, :3] * occ, occ], 1))
    x = torch.cat([_features(ctx, g) for g in pts.split(1 << 16)])
    return {"labels": torch.cat(out).cpu(), "features": torch.nn.functional.pad(x, (0, 31)).reshape(-1).cpu()}


def _layers(flat):
    """(W, b) of the four layers in the flat parameter vector."""
    out, o = [], 0
    for k, n in ((129, 64), (64, 64), (64, 64), (64, 3)):
        out.append((flat[o:o + n * k].reshape(n, k), flat[o + n * k:o + n * k + n]))
        o += n * k + n
    return out


def _network(flat, x):
    for i, (w, b) in enumerate(_layers(flat)):
        x = x @ w.T + b
        if i < 3:
            x = torch.relu(x)
    return x


def _exact_infer(st):
    ctx = st["ctx"]
    g, cov = _gbuffer(ctx)
    w = torch.from_numpy(ctx.weights()).double().to(g.device)
    out = torch.zeros(g.shape[0], 4, dtype=torch.float64, device=g.device)
    for at in cov.split(1 << 18):
        out[at, :3] = _network(w[:-1], _features(ctx, g[at])) * w[-1]
        out[at, 3] = 1.0
    return {"indirect": out.cpu()}


def _mix(x):
    x ^= x >> 16
    x = (x * 0x7FEB352D) & 0xFFFFFFFF
    x ^= x >> 15
    x = (x * 0x846CA68B) & 0xFFFFFFFF
    return x ^ (x >> 16)


def _exact_train(st):
    ctx, case = st["ctx"], st["case"]
    ctx.learned_train(steps=0, batch=case["batch"], lr=1e-3, seed=st["seed"], reset=True)
    first = torch.from_numpy(ctx.weights()).double().to(_dev())
    scale, w = first[-1], first[:-1].clone().requires_grad_()
    x = torch.from_numpy(ctx.download(abi.VCT_BUF_FEATURES, 0, np.int16)).view(torch.bfloat16).reshape(-1, 160)
    x = x[:, :129].to(_dev()).double()
    y = torch.from_numpy(ctx.download(abi.VCT_BUF_LABELS, 0, np.float32).reshape(-1, 4)[:, :3]).to(_dev()).double() / scale
    m, v, loss = torch.zeros_like(first[:-1]), torch.zeros_like(first[:-1]), []
    rows = np.arange(case["batch"], dtype=np.int64)
    for t in range(1, case["steps"] + 1):
        pick = torch.from_numpy(_mix(st["seed"] ^ _mix((t * 0x9E3779B9 + rows) & 0xFFFFFFFF)) % case["points"]).to(_dev())
        l = ((_network(w, x[pick]) - y[pick]) ** 2).mean()
        g, = torch.autograd.grad(l, w)
        loss.append(l.detach())
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        with torch.no_grad():
            w -= 1e-3 * (m / (1 - 0.9 ** t)) / (torch.sqrt(v / (1 - 0.999 ** t)) + 1e-8)
    return {"loss": torch.stack(loss).cpu(), "weights": torch.cat([w.detach(), first[-1:]]).cpu()}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("frame", "volume"):
        return None
    st = prepare(case, seed)
    if kind == "gather":
        return _exact_gather(st)
    if kind == "mip":
        return _exact_mip(st)
    if kind == "train":
        return _exact_train(st)
    if kind == "infer":
        return _exact_infer(st)
    return _exact_labels(st, seed)
