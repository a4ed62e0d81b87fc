"""The convolutions' tiles: every class of channel count (multiples of 64, of 32
and neither; the first layer's few), widths and heights that do not fill a
tile, and batches that take the larger tiles.  With two weights of +-1 per
output channel every sum is exact in FP32, so that forward outputs are the
oracle's (oracle/unet.py) bits; between batch sizes they are the same bits for
any weights (every output sums in the same order in every tile)."""
import importlib

import numpy as np
import pytest

from oracle import unet as U
from test_unet_grad_tiles_gpu import CIN, flat, setup, two_per_output

pytestmark = pytest.mark.gpu


def forward(P, x, base, cout):
    net = importlib.import_module("simple-ts_amd").UNet(CIN, cout, base, *x.shape[:3])
    net.set_params(flat(P, base, cout).astype(np.float32))
    return np.array(net.forward(x))


@pytest.mark.parametrize("base,N,H,W", [(8, 1, 8, 64), (16, 3, 24, 64), (24, 2, 16, 128), (32, 1, 40, 192),
                                        (40, 1, 24, 64), (64, 2, 8, 192), (96, 1, 16, 64)])
def test_forward_exact(base, N, H, W):
    print(f"U-Net forward base={base} {N}x{H}x{W}", flush=True)
    P, x, _ = setup(base, 2, N, H, W, 21)
    P, x = two_per_output(P, base, 2, 22), np.round(4 * x) / 4
    y, ref = forward(P, x, base, 2), U.UNet(P, CIN, 2, base).forward(x)
    assert np.array_equal(y, ref.reshape(y.shape)), np.abs(y - ref.reshape(y.shape)).max()


@pytest.mark.parametrize("base,N,H,W", [(8, 20, 64, 64), (32, 40, 64, 128), (64, 40, 72, 64)])
def test_forward_batches(base, N, H, W):
    print(f"U-Net forward base={base} {N}x{H}x{W}", flush=True)
    P, x, _ = setup(base, 2, 1, H, W, 23)
    one = forward(P, x, base, 2)
    many = forward(P, np.repeat(x, N, 0), base, 2).reshape(N, *one.shape[-3:])
    assert all(np.array_equal(many[k], one.reshape(many[k].shape)) for k in range(N))
