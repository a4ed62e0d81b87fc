"""Loop 2 at the sizes where the tiles of its kernels can go wrong: one cell
either side of a tile's width and height, grids smaller than a tile, grids
large enough for the larger tiles, both x boundary kinds and given velocities
at both ends.  FP64, bit-exact against the CPU restatement."""
import numpy as np
import pytest

from cases import bit_mismatch, channel_case, random_state

pytestmark = pytest.mark.gpu

SIZES = [(9, 9), (12, 61), (59, 10), (60, 11), (61, 12), (62, 13), (63, 9), (64, 17), (65, 16), (121, 14), (129, 15),
         (187, 100), (61, 390), (245, 121)]
KINDS = {
    "given_both": dict(given_xb=1, seed=2),
    "gravity_noslip": dict(given_xb=0, seed=3, gravity=0.5, kn_local=0, slip=(0, 0, 0, 0), jump=(0, 0, 0, 0),
                           bc=dict(dudx_0_xb=1, durhodx_0_xe=1, dvdx_0_xe=1, dvdy_0_ye=1, dpdx_0_xe=1, dTdy_0_yb=1)),
    "periodic": dict(given_xb=0, seed=4, periodic=True),
}


def _pair(sts, oracle, size, kind):
    prob = channel_case(Nx=size[0], Ny=size[1], **KINDS[kind])
    if kind == "given_both":
        prob.given_xe = 1
    ctx, ora = sts.Context(prob), oracle.Oracle(prob)
    for k, a in random_state(prob, seed=11).items():
        ctx.set(k, a)
        ora.set(k, a)
    return ctx, ora


def _same(sts, ctx, ora, names):
    bad = {n: bit_mismatch(ctx.get(n), ora.get(n)) for n in names}
    return {n: k for n, k in bad.items() if k}


@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("size", SIZES, ids=lambda s: f"{s[0]}x{s[1]}")
def test_two_sweep_pass(sts, oracle, size, kind):
    ctx, ora = _pair(sts, oracle, size, kind)
    rg, ro = ctx.pt_jacobi(4), ora.pt_jacobi(4)
    bad = _same(sts, ctx, ora, ("p", "Temper"))
    ctx.close()
    assert np.array_equal(rg, ro) and not bad, (rg, ro, bad)


@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("size", SIZES, ids=lambda s: f"{s[0]}x{s[1]}")
def test_loop_of_outer_iterations(sts, oracle, size, kind):
    """Three outer iterations inside one time step (the loops' own kernels,
    which keep Gamma and D out of memory) against three of the oracle's."""
    ctx, ora = _pair(sts, oracle, size, kind)
    ctx.fluxes_diffusion()
    ora.fluxes_diffusion()
    it, log, _ = ctx.time_step(3, 2, 0.0, 0.0, 0.0)
    ora.save_previous()
    ro = np.array([ora.outer_iteration(2) for _ in range(3)])
    bad = _same(sts, ctx, ora, sts.FIELDS)
    ctx.close()
    assert it == 3 and np.array_equal(log[:, :4], ro) and not bad, (log, ro, bad)


@pytest.mark.parametrize("depth", [1, 2, 3])
@pytest.mark.parametrize("size", [(130, 27), (1601, 257)], ids=["one_tile_each", "two_tiles_each"])
def test_anderson_mix_tiles(sts, size, depth, tmp_path):
    """Anderson steps on grids whose mix gives a workgroup one tile and two:
    both end on the reference's test, so the fields are the plain path's to
    the tolerance (1e-8) times the slow modes' amplification, as the other
    acceleration tests allow (1e-5 relative L2)."""
    import importlib

    ws = importlib.import_module("simple-ts_amd.warmstart")
    prm = dict(Ma=1.2, Kn=0.01, Re=1.2 / (0.01 * ws.SQ), side=0.25, xc=4.0)
    runs = [ws.Run(ws.write_case(str(tmp_path / n), *size, prm, 3, dt_over_tin=0.005 * 240 / size[0]))
            for n in ("plain", "aa")]
    n_plain = n_aa = 0
    for _ in range(2):
        n_plain += runs[0].step()
        n_aa += runs[1].ctx.time_step_mixed(*runs[1].loop, 0, (1e-7,) * 3, anderson=depth)[1]
    assert n_aa < n_plain, (n_aa, n_plain)
    for k in ("u", "v", "p", "Temper"):
        a, b = runs[0].ctx.get(k), runs[1].ctx.get(k)
        assert np.linalg.norm(a - b) <= 1e-5 * np.linalg.norm(a), k
    for r in runs:
        r.close()


@pytest.mark.parametrize("size", [(9, 9), (65, 16), (245, 121), (700, 90)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_loop_without_edge_conditions(sts, oracle, size):
    """No condition at any edge of the box: the wall writes then share the
    launch of the loop test and the probe; a few of them and several
    workgroups' worth."""
    prob = channel_case(Nx=size[0], Ny=size[1], seed=5, bc={})
    ctx, ora = sts.Context(prob), oracle.Oracle(prob)
    for k, a in random_state(prob, seed=11).items():
        ctx.set(k, a)
        ora.set(k, a)
    ctx.fluxes_diffusion()
    ora.fluxes_diffusion()
    it, log, _ = ctx.time_step(3, 2, 0.0, 0.0, 0.0)
    ora.save_previous()
    ro = np.array([ora.outer_iteration(2) for _ in range(3)])
    bad = _same(sts, ctx, ora, sts.FIELDS)
    ctx.close()
    assert it == 3 and np.array_equal(log[:, :4], ro) and not bad, (log, ro, bad)
