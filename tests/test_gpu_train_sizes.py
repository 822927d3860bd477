"""The training step at the sizes where its workgroups and partial sums have
edges: one workgroup, a number of partials below, at and past a multiple of 16,
fewer points than rows (rows repeat), the smallest point set.

Tolerances: the gradient's and the loss's of the full-size step (1e-3 and 1e-4
relative to the FP64 network with BF16 operands: FP32 sums and rare BF16
rounding flips apart)."""
import numpy as np
import pytest

from gpu_util import make_app, rel_err
from oracle import mlp_ref
from vct_amd import _abi as abi

pytestmark = pytest.mark.gpu


def _picks(seed, step, batch, npts):
    def mix(x):
        x = x ^ (x >> np.uint32(16))
        x = (x * np.uint32(0x7FEB352D)) & np.uint32(0xFFFFFFFF)
        x = x ^ (x >> np.uint32(15))
        x = (x * np.uint32(0x846CA68B)) & np.uint32(0xFFFFFFFF)
        return x ^ (x >> np.uint32(16))

    with np.errstate(over="ignore"):
        j = np.uint32(step * 0x9E3779B9 & 0xFFFFFFFF) + np.arange(batch, dtype=np.uint32)
        return mix(np.uint32(seed) ^ mix(j)) % np.uint32(npts)


@pytest.mark.parametrize("batch,npts", [(64, 64), (960, 1000), (1024, 64), (1088, 777)])
def test_training_step_sizes(batch, npts):
    app = make_app(1, dim=32)
    ctx = app.ctx
    app.build_radiance(0)
    ctx.learned_set_points(app.surface_points(npts, 0, seed=5))
    ctx.learned_prepare()
    lab = ctx.download(abi.VCT_BUF_LABELS, 0, np.float32).reshape(-1, 4)
    bits = ctx.download(abi.VCT_BUF_FEATURES, 0, np.uint16).astype(np.uint32) << 16
    X = bits.view(np.float32).reshape(-1, 160)[:, :129].astype(np.float64)
    scale = np.float32(max(np.abs(lab[:, :3].astype(np.float64)).mean(), 1e-6))
    rng = np.random.default_rng(batch)
    params = [(W, rng.normal(0, 0.05, b.shape)) for W, b in mlp_ref.init_params(3)]
    w = np.append(mlp_ref.flatten(params), scale).astype(np.float32)
    ctx.set_weights(w)
    loss_gpu = ctx.learned_train(steps=1, batch=batch, lr=1e-3, seed=9)
    grad = ctx.download(abi.VCT_BUF_GRADIENT, 0, np.float32)
    pick = _picks(9, 1, batch, npts)
    t = (lab[pick, :3] / scale).astype(np.float64)
    loss, grads = mlp_ref.loss_and_grads(mlp_ref.unflatten(w[:-1].astype(np.float64)), X[pick], t, bf16=True)
    assert abs(grad[-1] - loss) <= 1e-4 * loss and abs(loss_gpu[0] - loss) <= 1e-4 * loss
    gref = mlp_ref.flatten(grads)
    assert rel_err(grad[:-1], gref) < 1e-3, rel_err(grad[:-1], gref)
    g = grad[:-1].astype(np.float64)
    want = w[:-1].astype(np.float64) - 1e-3 * g / (np.abs(g) + 1e-8)
    assert np.abs(ctx.weights()[:-1] - want).max() < 1e-6
    app.close()
