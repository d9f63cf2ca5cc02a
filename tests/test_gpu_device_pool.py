"""Device memory kept between handles: graphs, plans and Bit-BSRs of many
sizes built and freed in turn, on several threads with a stream each and
with failing calls in between, count what the oracle counts."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _graphs(btc, seed):
    rng = np.random.default_rng(seed)
    out = []
    for k in range(6):
        n = int(rng.integers(40, 6000)) if k else 1
        e = int(n * rng.integers(1, 12))
        out.append((rng.integers(0, n, e).astype(np.int32), rng.integers(0, n, e).astype(np.int32), n))
    s, d = btc.gen_rmat(13, 8, seed=seed)
    out.append((s, d, 1 << 13))
    return out


def _run(btc, orc, seed, stream, errors):
    try:
        for rep in range(3):
            for s, d, n in _graphs(btc, seed + rep):
                g = btc.Graph.from_coo(s, d, n, btc.CANON_DEFAULT | btc.CANON_DEVICE)
                rp, col = g.csr()
                want, rows = orc.tc_merge(rp, col, threads=1, per_row=True)
                p = btc.Plan(g, planner=2, stream=stream)
                total, pv, _ = p.count(per_vertex=True, stream=stream)
                assert total == want and np.array_equal(pv, rows)
                with pytest.raises(btc.BtcError):  # id out of range: refused half-way
                    btc.Graph.from_coo(np.append(s, n), np.append(d, 0), n, btc.CANON_DEFAULT | btc.CANON_DEVICE)
                b = btc.BitBSR(g, 32, stream=stream)
                p.close()
                total, pv, _ = b.count(per_vertex=True, stream=stream)
                assert total == want and np.array_equal(pv, rows)
                b.close()
                g.close()
    except BaseException as e:  # noqa: BLE001 -- reported by the caller's thread
        errors.append(e)


@pytest.mark.parametrize("threads", [1, 4])
def test_reused_memory(gpu, orc, threads):
    hip = C.CDLL("libamdhip64.so")
    streams = [C.c_void_p() for _ in range(threads)]
    for s in streams:
        assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0
    errors = []
    work = [threading.Thread(target=_run, args=(gpu, orc, 100 * k, streams[k], errors)) for k in range(threads)]
    for t in work:
        t.start()
    for t in work:
        t.join()
    for s in streams:
        assert hip.hipStreamDestroy(s) == 0
    assert not errors, errors[0]
