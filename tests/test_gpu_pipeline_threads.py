"""Pipelines of several host threads at once: each stages its own pairs.

The staging teams share the cores while threads stage together, so a team of
any size from one thread up must still put every pair where it belongs: pair
counts lie around the smallest input that gets a team and around a staging
round, and each thread's totals are compared with the oracle's.
"""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PAIRS = [(1 << 15) - 1, (1 << 16) + 1, (1 << 19) + 5]


@pytest.mark.parametrize("threads", [2, 8])
def test_side_by_side(gpu, orc, threads):
    n = 20000
    inputs = []
    for k, e in enumerate(PAIRS):
        rng = np.random.default_rng(k)
        s, d = (rng.integers(0, n, e, dtype=np.int32) for _ in range(2))
        rp, col = gpu.Graph.from_coo(s, d, n).csr()
        inputs.append((s, d, orc.tc_merge(rp, col, threads=4)))
    pipes = [gpu.Pipeline(n, max(PAIRS)) for _ in range(threads)]
    start = threading.Barrier(threads)
    wrong = []

    def run(t):
        try:
            start.wait(60)
            for r in range(6):
                s, d, want = inputs[(t + r) % len(inputs)]
                got, _ = pipes[t].count(s, d, n)
                if got != want:
                    wrong.append((t, r, got, want))
        except Exception as err:
            wrong.append((t, repr(err)))
            start.abort()

    team = [threading.Thread(target=run, args=(t,)) for t in range(threads)]
    for t in team:
        t.start()
    for t in team:
        t.join()
    assert not wrong
