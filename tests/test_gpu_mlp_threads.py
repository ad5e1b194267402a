"""Networks trained by several threads at once: one pinned buffer per device stages host batches, and a thread that finds
it taken copies as before.  Every network ends with the bits it has when it trains alone."""
import threading

import numpy as np
import pytest

import orkan_amd
from orkan_amd import surrogate

pytestmark = pytest.mark.gpu


def _train(lib, k, out):
    rng = np.random.default_rng(k)
    m = surrogate.Mlp(lib, hidden=256, layers=2 + k % 2, max_batch=2048)
    m.init(rng)
    losses = []
    for step in range(40):
        rows = int(rng.integers(1, 2049))
        losses.append(m.train_step(rng.standard_normal((rows, 128)).astype(np.float32),
                                   rng.standard_normal(rows).astype(np.float32), 1e-3))
    out[k] = (losses, m.get_weights())
    m.close()


def test_threads_train_as_they_would_alone():
    lib = orkan_amd.load(5)
    alone, together = {}, {}
    for k in range(3):
        _train(lib, k, alone)
    threads = [threading.Thread(target=_train, args=(lib, k, together)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
    assert sorted(together) == [0, 1, 2]
    for k in range(3):
        (la, (Wa, ba, wa, oa)), (lb, (Wb, bb, wb, ob)) = alone[k], together[k]
        assert la == lb and oa == ob and np.array_equal(wa, wb)
        assert all(np.array_equal(x, y) for x, y in zip(Wa + ba, Wb + bb))
