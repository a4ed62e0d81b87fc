"""The weight gradients of the full-size level are the same bits from every tile
class, 32 x 32, 32 x 64 and 64 x 64 channels: with 32 x 64 pixels an image is one
run, so the sums of a batch of one image over and over (64 and 128 of it take the
wider tiles) are the FP32 sum, one after the other, of that image's own."""
import numpy as np
import pytest

from test_unet_grad_tiles_gpu import gradients, setup

pytestmark = pytest.mark.gpu

BASE, COUT, H, W = 64, 2, 32, 64


def test_tile_classes_agree():
    P, x, dy = setup(BASE, COUT, 1, H, W, 21)
    one = gradients(P, x, dy, BASE, COUT)
    for N in (64, 128):
        print(f"U-Net gradients of {N} equal images", flush=True)
        many = gradients(P, np.repeat(x, N, 0), np.repeat(dy, N, 0), BASE, COUT)
        again = gradients(P, np.repeat(x, N, 0), np.repeat(dy, N, 0), BASE, COUT)
        for k in many:
            assert np.array_equal(many[k], again[k]), k
        for k in ("e1a.w", "e1b.w", "d1a.w", "d1b.w"):
            s = np.zeros_like(one[k])
            for _ in range(N):
                s = s + one[k]
            assert np.array_equal(many[k], s), (N, k)
