"""Requests by key for graphs that were evicted before their results were
polled: accepted however late they come, answered exactly, and refused again
once every result has been polled."""
import time

import pytest

from test_gpu_serve import alone, drain, make_graphs, settled

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("captured", [0, 1])
def test_requests_by_key_after_eviction(gpu, orc, captured):
    gs = make_graphs(gpu, 24, seed=9)
    want = [alone(orc, *g) for g in gs]
    sv = gpu.Server(hbm_budget_bytes=2 << 20, max_batch=64, prep_threads=2, captured_prep=captured)
    ids = {}
    for k, g in enumerate(gs):
        ids[sv.submit(k, *g)] = k
        if k % 6 == 5:  # the next graphs find these resident and idle
            st = settled(sv, k + 1)
    assert st["prepared"] == 24 and st["evictions"] > 0
    time.sleep(0.1)  # longer than any preparation
    for order in (range(24), reversed(range(24))):
        ids.update({sv.submit(k): k for k in order})
        time.sleep(0.05)
    for r in drain(sv, len(ids)):
        assert r["status"] == 0 and r["triangles"] == want[ids[r["request_id"]]]
    # everything polled: an evicted graph has to be sent again
    got = {}
    for k in range(24):
        try:
            got[sv.submit(k)] = k
        except gpu.BtcError as e:
            assert e.code == 1
    assert len(got) < 24
    for r in drain(sv, len(got)):
        assert r["status"] == 0 and r["triangles"] == want[got[r["request_id"]]]
    st = sv.stats()
    assert st["failed"] == 0 and st["prepared"] == 24 and st["completed"] == 72 + len(got)
    again = {sv.submit(k, *g): k for k, g in enumerate(gs)}
    for r in drain(sv, 24):
        assert r["status"] == 0 and r["triangles"] == want[again[r["request_id"]]]
    sv.close()
