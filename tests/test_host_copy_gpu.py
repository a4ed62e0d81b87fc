"""Fields between host arrays and the device at the sizes where the copies'
pieces end: below one piece, one chunk and a little more, several chunks, more
than the pinned memory of a context; from several threads on one context; and a
network's inputs and outputs.  Exact: copies change no bit."""
import threading

import numpy as np
import pytest

from cases import channel_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(9, 9), (181, 181), (724, 724), (725, 724), (1024, 1025), (2060, 2050)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
def test_fields_round_trip(sts, size):
    ctx = sts.Context(channel_case(Nx=size[0], Ny=size[1], given_xb=0, seed=2))
    rng = np.random.default_rng(size[0])
    want = {k: rng.standard_normal(size[0] * size[1]) for k in ("u", "v", "p")}
    for k, a in want.items():
        ctx.set(k, a)
    got = {}

    def read(k):
        got[k] = [ctx.get(k) for _ in range(3)]

    threads = [threading.Thread(target=read, args=(k,)) for k in want]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    ctx.close()
    assert all(np.array_equal(b, want[k]) for k in want for b in got[k])


def test_network_arrays(sts):
    net = sts.UNet(9, 4, 8, 2, 512, 1024)  # 37.7 MB of inputs, 16.8 MB of outputs
    rng = np.random.default_rng(1)
    P = (0.05 * rng.standard_normal(net.n_params)).astype(np.float32)
    net.set_params(P)
    assert np.array_equal(net.get_params() if hasattr(net, "get_params") else net.params(), P)
    x = rng.standard_normal((2, 512, 1024, 9)).astype(np.float32)
    y = net.infer(x)
    halves = [net.infer(x[k:k + 1])[0] for k in range(2)]
    assert np.array_equal(y[0], halves[0]) and np.array_equal(y[1], halves[1])
