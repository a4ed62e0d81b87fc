"""The order of the parameter gradients' sums, and the training step as a whole.

Gradients of small networks whose activations are 1 and whose last hidden
layer's incoming gradient is dy itself, so that the last 3x3 layer's gradients
are sums of dy over the pixels: every run's sum is exact in FP32 and the total
shows the order of the runs.  A training step against the calls it stands for
on a network of the same parameters, and against itself: equal bits (the loss
to 1e-12: its FP64 sum is not in a fixed order)."""
import importlib

import numpy as np
import pytest

from oracle import unet as U

pytestmark = pytest.mark.gpu

BASE, CIN, COUT = 8, 5, 2


def in_order(parts):
    """FP32 sum of `parts` in turn."""
    s = np.float32(0)
    for p in parts:
        s = np.float32(s + np.float32(p))
    return s


@pytest.mark.parametrize("H", [72, 80, 88, 96])
def test_order_of_the_runs(H):
    """Behind two runs of 2048 pixels (the bias: four of 1024) one of 512, 1024, 1536
    or 2048 (one of 512; one of 1024; 1024 and 512; two of 1024)."""
    W = 64
    pkg = importlib.import_module("simple-ts_amd")
    net = pkg.UNet(CIN, 1, BASE, 1, H, W)
    P = {}
    for n, ci, co, k in U.conv_specs(CIN, 1, BASE):
        P[n + ".w"] = np.full((k * k, ci, co), 1.0 if n == "head" else 0.0, np.float32)
        P[n + ".b"] = np.full(co, 0.0 if n == "head" else 1.0, np.float32)
    net.set_params(np.concatenate([P[n + s].ravel() for n, _, _, _ in U.conv_specs(CIN, 1, BASE) for s in (".w", ".b")]))
    dy = np.full(H * W, 2.0 ** -23, np.float32)
    dy[:2048], dy[2048:4096] = 1.0, -1.0
    net.forward(np.zeros((1, H, W, CIN), np.float32))
    net.backward(dy.reshape(1, H, W, 1))
    v, o, G = net.grads(), 0, {}
    for n, ci, co, k in U.conv_specs(CIN, 1, BASE):
        G[n + ".w"] = v[o:o + k * k * ci * co].reshape(k * k, ci, co)
        G[n + ".b"] = v[o + k * k * ci * co:o + k * k * ci * co + co]
        o += (k * k * ci + 1) * co

    def total(run):
        sums = [in_order(dy[a:a + run]) for a in range(0, dy.size, run)]
        short = dy.size % run != 0 and dy.size % run <= 0.75 * run
        return in_order(sums[-1:] + sums[:-1] if short else sums)

    assert np.all(G["d1b.w"][4] == total(2048)), (G["d1b.w"][4, 0, 0], total(2048))  # tap 4: the pixel itself
    assert np.all(G["d1b.b"] == total(1024)), (G["d1b.b"][0], total(1024))


def training_set(net, run, n, seed):
    """Records n samples and gives the arrays they stand for."""
    pkg = importlib.import_module("simple-ts_amd")
    rng = np.random.default_rng(seed)
    net.dataset(n)
    xs, ts = [], []
    mask = (np.asarray(run.case.vol) == 0).reshape(net.H, net.W)
    for q in range(n):
        f = {k: 1.0 * (k in ("p", "Temper")) + 0.2 * rng.standard_normal((net.H, net.W))
             for k in ("u", "v", "p", "Temper")}
        t = {k: f[k] + 2e-3 * rng.standard_normal((net.H, net.W)) for k in ("p", "Temper")}
        for k in f:
            run.ctx.set(k + "_pr", f[k])
        for k in t:
            run.ctx.set(k, t[k])
        net.record(q, run.ctx, pkg.UNetNorm(1.0, 1.0, 2e-3, 2e-3))
        xs.append(np.stack([f["u"], f["v"], f["p"] - 1.0, f["Temper"] - 1.0, 1.0 * mask], -1).astype(np.float32))
        ts.append(np.stack([(t[k] - f[k]) * (1.0 / 2e-3) for k in ("p", "Temper")], -1).astype(np.float32))
    return np.stack(xs), np.stack(ts), np.stack(n * [mask])


@pytest.mark.parametrize("base,n,H,W", [(8, 2, 40, 64), (32, 3, 72, 128)])
def test_training_step_is_its_parts(base, n, H, W, tmp_path):
    ws = importlib.import_module("simple-ts_amd.warmstart")
    pkg = importlib.import_module("simple-ts_amd")
    print(f"training step base={base} {n}x{H}x{W}", flush=True)
    prm = dict(Ma=0.8, Kn=0.01, Re=0.8 / (0.01 * 0.6067627457812106), side=0.25, xc=4.0)
    run = ws.Run(ws.write_case(str(tmp_path / "c"), W, H, prm, 1))
    nets = [pkg.UNet(CIN, COUT, base, n, H, W) for _ in range(3)]
    for net in nets:
        net.set_params(ws.he_init(CIN, COUT, base, 3))
    x, t, m = [training_set(net, run, 2 * n, 17) for net in nets][-1]
    for step, slots in enumerate((list(range(n)), list(range(2 * n - 1, n - 1, -1)))):
        loss = [net.train_step(slots, 1e-3) for net in nets[:2]]
        nets[2].forward(x[slots])
        loss.append(nets[2].backward_mse(t[slots], m[slots]))
        nets[2].adam(1e-3)
        g, p = [net.grads() for net in nets], [net.params() for net in nets]
        for k in (1, 2):
            what = ("the same step again", "its parts")[k - 1]
            assert abs(loss[k] - loss[0]) <= 1e-12 * abs(loss[0]), (step, what, loss)
            assert np.array_equal(g[k], g[0]), (step, what, "gradients")
            assert np.array_equal(p[k], p[0]), (step, what, "parameters")
