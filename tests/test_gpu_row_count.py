"""The Bit-BSR count's row path at the edges of its classes and sets.

Row lengths around the cuts between 16-lane teams, waves and workgroups (64,
512) and the table and item sizes behind them (2048 ids, 256 lists), ids
inside and outside the LDS window of each team (8192, 32768 and 131072 ids),
lists long enough to be searched, and thresholds that send no tile, some
tiles or every tile down the dense path.  Counts are integers: equality.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rows_graph(lengths, spread, seed):
    """Row n0 + k holds lengths[k] distinct ids below n0 = spread, among them
    rows of a random base graph, so that many pairs close triangles."""
    rng = np.random.default_rng(seed)
    n0 = spread
    hubs = rng.choice(n0, size=min(n0, 4000), replace=False)
    s = [rng.choice(hubs, 30000)]
    d = [rng.choice(hubs, 30000)]
    for k, m in enumerate(lengths):
        pool = hubs if m <= hubs.size // 2 else np.arange(n0)
        ids = rng.choice(pool, size=m, replace=False)
        s.append(np.full(m, n0 + k))
        d.append(ids)
    # a few rows above join the long ones, so that a short row meets long lists
    top = n0 + len(lengths)
    for k in range(40):
        pick = rng.choice(len(lengths), size=min(len(lengths), 3 + k % 5), replace=False)
        s.append(np.full(pick.size, top + k))
        d.append(n0 + pick)
        extra = rng.choice(hubs, size=2 + k, replace=False)
        s.append(np.full(extra.size, top + k))
        d.append(extra)
    return np.concatenate(s).astype(np.int32), np.concatenate(d).astype(np.int32), top + 40


def check(btc, orc, s, d, n, K, taus, flags=0):
    g = btc.Graph.from_coo(s, d, n, flags)
    rp, col = g.csr()
    want, rows = orc.tc_merge(rp, col, per_row=True)
    b = btc.BitBSR(g, K)
    for tau in taus:
        for mfma in (False, True):
            t, pv, _ = b.count(tau=tau, per_vertex=True, mfma=mfma)
            assert t == want, (K, tau, mfma, t, want)
            assert np.array_equal(pv, rows), (K, tau, mfma)
            t, _, _ = b.count(tau=tau, mfma=mfma)
            assert t == want
    b.close()
    g.close()


@pytest.mark.parametrize("K", [32, 64, 128])
@pytest.mark.parametrize("spread", [8100, 8191, 8192, 8300, 32760, 32800, 131000, 131200])
def test_row_classes_and_windows(gpu, orc, K, spread):
    lengths = [0, 1, 2, 3, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 768, 1023, 2047, 2048, 2049, 4100]
    s, d, n = rows_graph(lengths, spread, spread + K)
    check(gpu, orc, s, d, n, K, [-1, 8])


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 33, 100, 129])
@pytest.mark.parametrize("K", [32, 64, 128])
def test_complete_graphs(gpu, orc, n, K):
    u, v = np.triu_indices(n, 1)
    check(gpu, orc, u.astype(np.int32), v.astype(np.int32), n, K, [-1, 0, 40, 16 * K])


def test_light_rows_mixed_in_a_wave(gpu, orc):
    """Neighbouring rows with and without a window, of very different lengths."""
    rng = np.random.default_rng(5)
    n = 60000
    s, d = [], []
    for i in range(40000, 42000):
        m = int(rng.integers(0, 65))
        near = rng.integers(0, 2) == 0
        lo = i - 300 if near else 0
        ids = rng.choice(np.arange(lo, i), size=min(m, i - lo), replace=False)
        s.append(np.full(ids.size, i))
        d.append(ids)
    check(gpu, orc, np.concatenate(s).astype(np.int32), np.concatenate(d).astype(np.int32), n, 64, [-1])


def test_no_triangles_and_no_edges(gpu, orc):
    e = np.zeros(0, np.int32)
    check(gpu, orc, e, e, 50, 32, [-1, 0])
    check(gpu, orc, np.arange(1, 3000, dtype=np.int32), np.zeros(2999, np.int32), 3000, 128, [-1, 0])
