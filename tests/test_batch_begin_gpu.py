"""The start of a step of all cases of a batch at once -- previous fields,
history, predicted starts and the fields derived from them -- for every cell
tile, with cases that predict beside cases that do not: the single contexts'
counts and fields, bit for bit."""
import importlib

import numpy as np
import pytest

from test_batch_gpu import runs, state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", range(4))
def test_starts_of_a_batch(variant, tmp_path):
    pkg = importlib.import_module("simple-ts_amd")
    single, batched = runs(tmp_path, "s"), runs(tmp_path, "b")
    loop = single[0].loop
    acc = (0, (1e-7,) * 3, 0, 0.95)
    for r in (single[0], batched[0]):  # a history of two steps that the other cases do not have
        for _ in range(2):
            r.ctx.time_step_mixed(*loop, *acc, extrapolate=3)
    B = pkg.Batch([r.ctx for r in batched])
    B.set_tiles(variant, variant)
    for _ in range(4):
        ref = [r.ctx.time_step_mixed(*loop, *acc, extrapolate=3)[1] for r in single]
        assert B.time_step(*loop, mixed=acc + (3,))[1] == ref
    B.close()
    for a, b in zip(single, batched):
        for x, y in zip(state(a), state(b)):
            assert np.array_equal(x, y)
    for r in single + batched:
        r.close()
