"""The FP32 instances of the loop's kernels at the sizes where their tiles can go
wrong: three FP32 outer iterations and one in FP64 against four of the CPU
restatement, which is FP64.

Tolerance: an FP32 iteration rounds some 100 operations per cell, of terms at most
about ten times the fields (coefficients of neighbours up to 1.5, pressure
differences up to 0.8), at 2^-24 each: at most 100 * 10 * 6e-8 = 6e-5 if every
rounding went the same way, about 6e-6 at random signs.  Three iterations, each a
contraction in p and T and an update of u, v by terms of the order of the fields:
three times that, below 1e-4 (absolute; the fields are of order one).  A mesh
step or reciprocal of the wrong cell is off by 10 % and more here."""
import numpy as np
import pytest

from cases import channel_case, random_state

pytestmark = pytest.mark.gpu

SIZES = [(9, 9), (59, 10), (61, 12), (64, 17), (65, 16), (130, 15), (245, 121), (449, 121), (705, 137)]


@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("size", SIZES, ids=lambda s: f"{s[0]}x{s[1]}")
def test_fp32_iterations(sts, oracle, size, periodic):
    prob = channel_case(Nx=size[0], Ny=size[1], given_xb=0, seed=5, gravity=0.3, periodic=periodic)
    rng = np.random.default_rng(7)
    prob.hx *= rng.uniform(0.7, 1.4, prob.hx.shape)
    prob.hy *= rng.uniform(0.7, 1.4, prob.hy.shape)
    print("FP32", size, periodic, flush=True)
    ctx, ora = sts.Context(prob, 32), oracle.Oracle(prob)
    for k, a in random_state(prob, seed=12).items():
        ctx.set(k, a)
        ora.set(k, a)
    ctx.fluxes_diffusion()
    ora.fluxes_diffusion()
    n32, n64, log, _ = ctx.time_step_mixed(1, 2, 0.0, 0.0, 0.0, 3, (0.0, 0.0, 0.0), stall_w=0)
    ora.save_previous()
    ro = np.array([ora.outer_iteration(2) for _ in range(4)])
    assert (n32, n64) == (3, 1)
    worst = {k: float(np.max(np.abs(ctx.get(k) - ora.get(k)))) for k in ("u", "v", "p", "Temper", "rho", "Fx", "Fy")}
    ctx.close()
    e = np.abs(log[:, :4] - ro)
    print("worst", worst, "residuals", e.max(), flush=True)
    assert e.max() <= 1e-4 and max(worst.values()) <= 1e-4, (worst, log, ro)
