"""GPU MLP kernels (forward, backward, loss, Adam) against the float64
oracle. Bar: fp32 forward within 1e-4 relative of the output scale,
gradients within 1e-3 relative of each tensor's scale (fp32 accumulation
over the batch), Adam update within 1e-6."""
import ctypes

import numpy as np
import pytest
import torch

from ipc_warp_amd import warmstart
from oracle import mlp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 37, 3000])
def test_forward_backward_match_oracle(dev, n):
    rng = np.random.default_rng(n)
    p = mlp.init(3)
    x = rng.standard_normal((n, mlp.IN)).astype(np.float32)
    t = rng.standard_normal((n, mlp.OUT)).astype(np.float32)
    w = rng.random(n).astype(np.float32) + 0.5
    net = warmstart.MLP(dev, params=torch.from_numpy(p.astype(np.float32)).to(dev))
    xt = torch.from_numpy(x).to(dev)
    y, work = net.forward(xt, keep=True)
    loss, dy = net.mse(y, torch.from_numpy(t).to(dev), torch.from_numpy(w).to(dev))
    grad = torch.zeros_like(net.params)
    net.backward(xt, work, dy, grad)
    torch.cuda.synchronize()
    yr, cache = mlp.forward(p.astype(np.float32).astype(np.float64), x.astype(np.float64))
    lr_, dyr = mlp.mse(yr, t.astype(np.float64), w.astype(np.float64))
    gr = mlp.backward(p.astype(np.float32).astype(np.float64), cache, dyr)
    yg = y.cpu().numpy()
    assert np.abs(yg - yr).max() <= 1e-4 * max(1.0, np.abs(yr).max())
    assert loss == pytest.approx(lr_, rel=1e-4)
    gg = grad.cpu().numpy().astype(np.float64)
    o = 0
    for name, shape in mlp.SHAPES:
        k = int(np.prod(shape))
        a, b = gg[o:o + k], gr[o:o + k]
        assert np.abs(a - b).max() <= 1e-3 * max(1e-6, np.abs(b).max()), name
        o += k


def test_adam_step_matches_oracle(dev):
    rng = np.random.default_rng(5)
    n = 10007
    p, g = rng.standard_normal(n), rng.standard_normal(n)
    m, v = rng.standard_normal(n) * 0.1, rng.random(n) * 0.1
    pt, gt, mt, vt = (torch.from_numpy(a.astype(np.float32)).to(dev) for a in (p, g, m, v))
    warmstart.adam_step(pt, gt, mt, vt, lr=1e-3, step=7)
    torch.cuda.synchronize()
    pr, mr, vr = mlp.adam(p.astype(np.float32).astype(np.float64), g.astype(np.float32).astype(np.float64),
                          m.astype(np.float32).astype(np.float64), v.astype(np.float32).astype(np.float64),
                          1e-3, 0.9, 0.999, 1e-8, 7)
    assert np.abs(pt.cpu().numpy() - pr).max() <= 1e-6
    assert np.abs(mt.cpu().numpy() - mr).max() <= 1e-6


def test_training_reduces_loss(dev):
    rng = np.random.default_rng(6)
    n = 4096
    x = rng.standard_normal((n, mlp.IN)).astype(np.float32)
    A = rng.standard_normal((mlp.IN, mlp.OUT)) * 0.3
    t = (np.tanh(x @ A)).astype(np.float32)
    net = warmstart.MLP(dev, seed=0)
    xt, tt = torch.from_numpy(x).to(dev), torch.from_numpy(t).to(dev)
    first = net.train_epochs(xt, tt, None, epochs=1, batch=1024, lr=1e-3)
    last = net.train_epochs(xt, tt, None, epochs=30, batch=1024, lr=1e-3)
    assert last < 0.2 * first


@pytest.mark.parametrize("n", [16, 17, 63, 65, 255, 257, 4097, 8191, 8192, 8209])
def test_row_tiles_and_splits_match_oracle(dev, n):
    """Rows around the tiles of 16, 32 and 64, the gradient's row splits (256
    a split, at most 16) and the change from 16 to 32 rows a workgroup at
    8192. A sum of n products in fp32 is off by at most n 2^-24 of the sum of
    their magnitudes; typical sums by its square root, and the bars leave ten
    times that."""
    rng = np.random.default_rng(n)
    p = mlp.init(4).astype(np.float32)
    x = rng.standard_normal((n, mlp.IN)).astype(np.float32)
    dy = rng.standard_normal((n, mlp.OUT)).astype(np.float32)
    net = warmstart.MLP(dev, params=torch.from_numpy(p).to(dev))
    xt = torch.from_numpy(x).to(dev)
    y, work = net.forward(xt, keep=True)
    y2, _ = net.forward(xt)
    grad = torch.zeros_like(net.params)
    net.backward(xt, work, torch.from_numpy(dy).to(dev), grad)
    torch.cuda.synchronize()
    yr, cache = mlp.forward(p.astype(np.float64), x.astype(np.float64))
    gr = mlp.backward(p.astype(np.float64), cache, dy.astype(np.float64))
    assert torch.equal(y, y2)
    assert np.abs(y.cpu().numpy() - yr).max() <= 10 * 2.0 ** -24 * 16 * np.abs(yr).max()
    kept = work.cpu().numpy().reshape(6, n, mlp.HID)
    for k in range(6):
        assert np.abs(kept[k] - cache[1 + k]).max() <= 10 * 2.0 ** -24 * 16 * np.abs(cache[1 + k]).max()
    gg = grad.cpu().numpy().astype(np.float64)
    o = 0
    for name, shape in mlp.SHAPES:
        k = int(np.prod(shape))
        a, b = gg[o:o + k], gr[o:o + k]
        assert np.linalg.norm(a - b) <= 10 * 2.0 ** -24 * np.sqrt(max(n, 256)) * np.linalg.norm(b), name
        o += k


def _gelu_and_derivative(dev, z):
    """gelu(z) from a forward pass (H1 with W1 = 0, b1 = z) and gelu'(z) from
    a backward pass of one row (db3 with Z3 = z, dy W4 = 1), 256 at a time."""
    at, o = {}, 0
    for name, shape in mlp.SHAPES:
        at[name] = slice(o, o + int(np.prod(shape)))
        o = at[name].stop
    g, d = np.empty_like(z), np.empty_like(z)
    x = torch.zeros((1, mlp.IN), device=dev)
    for k in range(0, z.size, 256):
        p = np.zeros(o, np.float32)
        p[at["b1"]] = z[k:k + 256]
        p[at["W4"]][:256] = 1
        net = warmstart.MLP(dev, params=torch.from_numpy(p).to(dev))
        _, work = net.forward(x, keep=True)
        g[k:k + 256] = work[256:512].cpu().numpy()
        work = torch.zeros(6 * 256, device=dev)
        work[4 * 256:5 * 256] = torch.from_numpy(z[k:k + 256]).to(dev)
        grad = torch.zeros_like(net.params)
        net.backward(x, work, torch.tensor([[1.0, 0.0, 0.0]], device=dev), grad)
        d[k:k + 256] = grad[at["b3"]].cpu().numpy()
    return g, d


def test_gelu_and_derivative_errors(dev):
    """No further from the fp64 values than 0.5 z (1 + erff) and 0.5 (1 + erff)
    + z phi with expf are in fp32: measured over these z, gelu 2.50e-8 rms and
    2.8e-7 at most, the derivative 2.73e-8 and 1.43e-7; over [-4, 0] 2.2e-8 and
    1.3e-8 rms. Infinities and NaN as those formulas give."""
    rng = np.random.default_rng(1)
    normal = rng.standard_normal(65536).astype(np.float32)
    lower = rng.uniform(-4, 0, 16384).astype(np.float32)
    for z, g_rms, g_max, d_rms, d_max in ((normal, 2.50e-8, 2.8e-7, 2.73e-8, 1.43e-7),
                                          (lower, 2.2e-8, 6.1e-8, 1.31e-8, 7e-8)):
        g, d = _gelu_and_derivative(dev, z)
        eg, ed = g - mlp.gelu(z.astype(np.float64)), d - mlp.gelu_grad(z.astype(np.float64))
        print(f"gelu {np.sqrt((eg ** 2).mean()):.2e} {np.abs(eg).max():.2e} "
              f"derivative {np.sqrt((ed ** 2).mean()):.2e} {np.abs(ed).max():.2e}", flush=True)
        assert np.sqrt((eg ** 2).mean()) <= g_rms and np.abs(eg).max() <= g_max
        assert np.sqrt((ed ** 2).mean()) <= d_rms and np.abs(ed).max() <= d_max
    z = np.zeros(256, np.float32)
    z[:9] = [np.inf, -np.inf, np.nan, 0.0, -0.0, 1e30, -1e30, 20.0, -20.0]
    g, d = _gelu_and_derivative(dev, z)
    assert np.array_equal(g[:9], np.array([np.inf, np.nan, np.nan, 0, 0, 1e30, 0, 20, 0], np.float32), equal_nan=True)
    assert np.array_equal(d[:9], np.array([np.nan, np.nan, np.nan, 0.5, 0.5, 1, 0, 1, 0], np.float32), equal_nan=True)


@pytest.mark.parametrize("n", [4096, 8192, 8193, 8240, 8241, 8256, 8257, 32768, 121904])
def test_large_batch_gradient_sums(dev, n):
    """Batches around 128 tiles of 64 rows (past them layer 1 is summed in a
    launch of its own, a last tile of 48 rows and fewer by atomics), and large
    ones, with positive x and dy so that the sums grow: against fp64 sums of
    the kept activations. A sum's at most 128 fp32 adders each round by
    2^-24 / sqrt(3) of the sum so far, rms: in all 2^-24 sqrt(128) / 3 = 2.2e-7,
    and a tile's own terms 3e-8."""
    rng = np.random.default_rng(n)
    net = warmstart.MLP(dev, params=torch.from_numpy(mlp.init(4).astype(np.float32)).to(dev))
    x = torch.from_numpy(np.abs(rng.standard_normal((n, mlp.IN))).astype(np.float32)).to(dev)
    dy = torch.from_numpy(np.abs(rng.standard_normal((n, mlp.OUT))).astype(np.float32)).to(dev)
    _, work = net.forward(x, keep=True)
    grad = torch.zeros_like(net.params)
    net.backward(x, work, dy, grad)
    W, at, o = {}, {}, 0
    for name, shape in mlp.SHAPES:
        at[name] = slice(o, o + int(np.prod(shape)))
        W[name] = net.params[at[name]].double().view(shape)
        o = at[name].stop
    Z1, H1, Z2, H2, Z3, H3 = (w.double() for w in work.view(6, n, mlp.HID))
    D = dy.double()

    def slope(z):
        return 0.5 * torch.erfc(-z / 2 ** 0.5) + z * torch.exp(-0.5 * z * z) / (2 * np.pi) ** 0.5

    d3 = (D @ W["W4"]) * slope(Z3)
    d2 = (d3 @ W["W3"]) * slope(Z2)
    d1 = (d2 @ W["W2"]) * slope(Z1)
    want = {"W4": D.T @ H3, "b4": D.sum(0), "W3": d3.T @ H2, "b3": d3.sum(0), "W2": d2.T @ H1, "b2": d2.sum(0),
            "W1": d1.T @ x.double(), "b1": d1.sum(0)}
    for name, w in want.items():
        err = float((grad[at[name]].double() - w.reshape(-1)).norm() / w.norm())
        print(f"{name} {err:.2e}", end=" ", flush=True)
        assert err <= 2.5e-7, name


def test_inference_allocates_its_output_only(dev):
    net = warmstart.MLP(dev)
    x = torch.zeros((20000, mlp.IN), device=dev)
    net.forward(x)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    y, _ = net.forward(x)
    assert torch.cuda.max_memory_allocated() - before <= y.numel() * 4 + 512
