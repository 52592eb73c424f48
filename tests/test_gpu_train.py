"""The MLP root's loss and gradients at the edges of the kernel's tiles (64 samples a wave, 1024
a block, 256 blocks before a wave takes a second tile), against a float64 restatement."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


@pytest.mark.parametrize("h", [8, 16, 32, 64])
@pytest.mark.parametrize("count", [1, 63, 64, 65, 1023, 1024, 1025, 5000, 262_144, 262_145, 600_001])
def test_loss_and_gradients(gj, gpu, h, count):
    rng = np.random.default_rng(h * count)
    edges = np.linspace(0, 1, h + 1)
    w1 = (h * (1 + 0.1 * rng.random(h))).astype(np.float32)
    b1 = (-edges[:h] * w1).astype(np.float32)
    w2 = ((1 + 0.1 * rng.random(h)) / h).astype(np.float32)
    b2 = np.float32(0.01)
    x = rng.random(count).astype(np.float32)
    x[0] = 0.0  # sits on the first ramp's foot, which passes no gradient
    y = (x * x * (3 - 2 * x)).astype(np.float32)

    f64 = np.float64
    a = (x[:, None].astype(f64) * w1 + b1).astype(np.float32)  # the kernel's FP32 fma
    ramp = np.clip(a, 0, 1).astype(f64)
    r = ramp @ w2.astype(f64) + f64(b2) - y
    g = 2.0 * r / count
    on = (a > 0) & (a < 1)
    gx = np.where(on, g[:, None] * x[:, None], 0.0)
    terms = [gx * w2, np.where(on, g[:, None], 0.0) * w2, g[:, None] * ramp]
    want = np.concatenate([t.sum(0) for t in terms] + [[g.sum()]])
    size = np.concatenate([np.abs(t).sum(0) for t in terms] + [[np.abs(g).sum()]])
    # f: H + 1 fused steps on values up to sum w2 + b2, then f - y; every term carries that error of g;
    # sums: at most 64 FP32 additions in a wave and 256 between blocks, a few roundings a term
    err_f = (h + 3) * EPS * (w2.sum(dtype=f64) + f64(b2) + 1)
    weight = np.concatenate([(on * x[:, None]).sum(0) * w2, on.sum(0) * w2, ramp.sum(0), [count]])
    tol = (64 + 256 + 8) * EPS * size + 2.0 / count * err_f * weight

    dev = [gj.DeviceArray.from_numpy(v) for v in (np.concatenate([w1, b1, w2, [b2]]).astype(np.float32), x, y)]
    grad, loss = gj.DeviceArray(3 * h + 1, np.float32), gj.DeviceArray(1, np.float32)
    grad.fill(0x5A)
    loss.fill(0x5A)
    for _ in range(2):  # a second call starts from zero again
        gj.mlp_loss_grad(dev[0], h, dev[1], dev[2], grad, loss)
    gj.synchronize()
    assert (np.abs(grad.numpy() - want) <= tol).all()
    want_loss = (r * r).mean()
    tol_loss = 264 * EPS * want_loss + 2 * err_f * np.abs(r).mean() + err_f ** 2
    assert abs(float(loss.numpy()[0]) - want_loss) <= tol_loss
