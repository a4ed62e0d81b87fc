"""Every condition at the x ends of the box, alone and beside one at the other
end, in the loops' form (u, v, temperature and pressure side by side, both ends
of a direction together, the fluxes of the cells they change formed again), on
an ordinary grid, one whose box is one column wide, and one with more rows than
a workgroup has threads.  FP64, bit-exact against the CPU restatement."""
import numpy as np
import pytest

from cases import bit_mismatch, channel_case, random_state

pytestmark = pytest.mark.gpu

KINDS = [("u_Min_Mout_xe",), ("u_Min_Mout_xe", "dudx_0_xb"), ("u_Min_Mout_xe", "durhodx_0_xb", "dvdx_0_xe"),
         ("durhodx_0_xb", "durhodx_0_xe"), ("dudx_0_xb", "dudx_0_xe"), ("drhodt_xb", "dvdx_0_xb"),
         ("drhodt_xe", "drhodt_xb", "dvdy_0_yb"), ("drhodt_xe", "dudx_0_xb", "dudy_0_ye")]


@pytest.mark.parametrize("kinds", KINDS, ids="+".join)
@pytest.mark.parametrize("size", [(40, 16), (4, 12), (20, 1100)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_edge_kinds(sts, oracle, size, kinds):
    Nx, Ny = size
    c = channel_case(Nx=max(Nx, 12), Ny=Ny, seed=3)
    vol = c.vol.reshape(Ny, -1)[:, :Nx].copy()
    if Nx < 12:  # no bodies between the walls
        vol[1:-1] = 0
    if "u_Min_Mout_xe" in kinds:  # it divides by the last row's face density
        vol[-1] = 0
    boxes = dict(c.boxes, Nx_u=(1, Nx - 1), Nx_v=(1, Nx - 2), Nx_o=(1, Nx - 2))
    bc = dict({k: 1 for k in kinds}, dTdx_0_xe=1, dpdx_0_xb=1)
    prob = sts.Problem(c.hx[:Nx], c.hy, vol, c.bodies, boxes, c.scalars, kn_local=1, bc=bc)
    print("edges", size, kinds, flush=True)
    ctx, ora = sts.Context(prob), oracle.Oracle(prob)
    for k, a in random_state(prob, seed=11).items():
        ctx.set(k, a)
        ora.set(k, a)
    ctx.fluxes_diffusion()
    ora.fluxes_diffusion()
    it, log, _ = ctx.time_step(3, 2, 0.0, 0.0, 0.0)
    ora.save_previous()
    ro = np.array([ora.outer_iteration(2) for _ in range(3)])
    bad = {n: bit_mismatch(ctx.get(n), ora.get(n)) for n in sts.FIELDS}
    bad = {n: k for n, k in bad.items() if k}
    ctx.close()
    assert it == 3 and np.all(np.isfinite(ro)) and np.array_equal(log[:, :4], ro) and not bad, (log, ro, bad)
