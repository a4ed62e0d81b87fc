"""The two-sweep pass either side of the line between its tiles of 2 rows (at most
512 of them) and of 6, one cell more or less than whole tiles.  FP64, bit-exact
against the CPU restatement."""
import numpy as np
import pytest

from cases import bit_mismatch, channel_case, random_state

pytestmark = pytest.mark.gpu

SIZES = [(480, 128), (480, 129), (481, 114), (659, 95), (660, 96), (661, 97), (59, 1026), (61, 515)]


@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("size", SIZES, ids=lambda s: f"{s[0]}x{s[1]}")
def test_sweep_rows(sts, oracle, size, periodic):
    prob = channel_case(Nx=size[0], Ny=size[1], given_xb=0, seed=6, periodic=periodic)
    ctx, ora = sts.Context(prob), oracle.Oracle(prob)
    for k, a in random_state(prob, seed=13).items():
        ctx.set(k, a)
        ora.set(k, a)
    rg, ro = ctx.pt_jacobi(4), ora.pt_jacobi(4)
    bad = {n: bit_mismatch(ctx.get(n), ora.get(n)) for n in ("p", "Temper")}
    ctx.close()
    assert np.array_equal(rg, ro) and not any(bad.values()), (rg, ro, bad)
