"""Four contexts, each stepped by its own thread, all threads on one processor:
while one waits for its loop another gets the processor, so that together they
take less than one after the other (0.7 times at 960 x 192; 1.0 to 1.4 times when
the wait keeps the processor)."""
import importlib
import os
import threading
import time

import pytest

pytestmark = pytest.mark.gpu


def test_waiting_contexts_share_a_processor(tmp_path):
    ws = importlib.import_module("simple-ts_amd.warmstart")
    prm = dict(Ma=1.2, Kn=0.01, Re=1.2 / (0.01 * ws.SQ), side=0.25, xc=4.0)
    runs = [ws.Run(ws.write_case(str(tmp_path / str(n)), 960, 192, prm, 1)) for n in range(4)]
    for r in runs:
        r.step()
    cpu = min(os.sched_getaffinity(0))

    def steps(r):
        os.sched_setaffinity(0, {cpu})  # (of this thread)
        for _ in range(6):
            r.step()

    def together(rs):
        t = [threading.Thread(target=steps, args=(r,)) for r in rs]
        a = time.perf_counter()
        for x in t:
            x.start()
        for x in t:
            x.join()
        return time.perf_counter() - a

    alone = [together([r]) for r in runs]
    both = together(runs)
    print(f"alone {[round(a * 1e3, 1) for a in alone]} ms, together {both * 1e3:.1f} ms", flush=True)
    for r in runs:
        r.close()
    assert both <= 0.95 * sum(alone)
