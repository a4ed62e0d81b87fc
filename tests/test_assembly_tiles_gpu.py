"""The loops' assembly on grids that take each of its tiles (64 x 2 and 64 x 4
with three threads per cell, 64 x 8 with one), with incomplete last columns and
rows of tiles, and with mesh steps that vary from cell to cell, so that every
quotient formed from a reciprocal has another divisor.  FP64, bit-exact against
the CPU restatement."""
import numpy as np
import pytest

from cases import bit_mismatch, channel_case, random_state

pytestmark = pytest.mark.gpu

SIZES = [(63, 10), (64, 13), (65, 12), (130, 15), (449, 121), (448, 126), (511, 125), (705, 137), (640, 136)]


@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("size", SIZES, ids=lambda s: f"{s[0]}x{s[1]}")
def test_assembly_tiles(sts, oracle, size, periodic):
    prob = channel_case(Nx=size[0], Ny=size[1], given_xb=0, seed=5, gravity=0.3, periodic=periodic)
    rng = np.random.default_rng(7)
    prob.hx *= rng.uniform(0.7, 1.4, prob.hx.shape)
    prob.hy *= rng.uniform(0.7, 1.4, prob.hy.shape)
    ctx, ora = sts.Context(prob), oracle.Oracle(prob)
    for k, a in random_state(prob, seed=12).items():
        ctx.set(k, a)
        ora.set(k, a)
    ctx.fluxes_diffusion()
    ora.fluxes_diffusion()
    it, log, _ = ctx.time_step(2, 1, 0.0, 0.0, 0.0)
    ora.save_previous()
    ro = np.array([ora.outer_iteration(1) for _ in range(2)])
    bad = {n: bit_mismatch(ctx.get(n), ora.get(n)) for n in sts.FIELDS}
    bad = {n: k for n, k in bad.items() if k}
    ctx.close()
    assert it == 2 and np.array_equal(log[:, :4], ro) and not bad, (log, ro, bad)
