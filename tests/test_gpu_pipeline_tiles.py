"""The captured build's tile passes at their edges: pair counts around one
and several tiles of every pass, for small capacities (tiles of 512) and
large ones (2048), each run on a replayed graph after runs of other sizes;
L, labels and counts equal the host canonicalisation's and the oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pairs(rng, n, e, kind):
    if kind == "random":
        return rng.integers(0, n, e), rng.integers(0, n, e)
    if kind == "star":  # one hub in every pair: one row, one degree counter
        return np.full(e, n - 1), rng.integers(0, n, e)
    return np.full(e, 3 % n), np.full(e, 1 % n)  # one pair, repeated


@pytest.mark.parametrize("flags", [0, 1, 2, 3])
@pytest.mark.parametrize("e_cap", [1 << 13, 1 << 19])
def test_tile_edges(gpu, orc, e_cap, flags):
    n_cap = 1 << 14
    p = gpu.Pipeline(n_cap, e_cap, flags)
    rng = np.random.default_rng(e_cap + flags)
    tile = 512 if e_cap <= 1 << 18 else 2048
    sizes = [0, 1, 2, 3, 5, tile - 1, tile, tile + 1, 2 * tile, 3 * tile + 7, min(e_cap, 40 * tile)]
    for k, e in enumerate(sizes + sizes[::-1]):
        n = int(rng.choice([1, 2, 64, 300, 5000, n_cap]))
        kind = ("random", "star", "same")[k % 3]
        s, d = (x.astype(np.int32) for x in _pairs(rng, n, e, kind))
        host = gpu.Graph.from_coo(s, d, n, flags)
        rp, col = host.csr()
        total, _ = p.count(s, d, n)
        q = p.graph()
        rp2, col2 = q.csr()
        assert np.array_equal(rp, rp2) and np.array_equal(col, col2), (e, n, kind)
        assert np.array_equal(host.labels(), q.labels()), (e, n, kind)
        assert total == orc.tc_merge(rp, col, threads=4), (e, n, kind)


@pytest.mark.parametrize("k", [1, 2, 63, 64])
def test_group_ranges_on_the_device(gpu, orc, k):
    """Several graphs whose ids are checked and moved by the device: empty
    graphs, ranges taken from the pairs (n <= 0), arrays on both sides of a
    staging piece; a refused call names the first bad graph and leaves the
    last run's batch exportable."""
    rng = np.random.default_rng(k)
    p = gpu.Pipeline(1 << 17, 1 << 19, 3, max_graphs=64)
    gs = []
    for g in range(k):
        n = int(rng.integers(1, 1500))
        e = 0 if g % 7 == 3 else int(rng.integers(1, 6 * n + 2))
        if g == 1:
            n, e = 4000, (1 << 16) + 5
        s, d = (rng.integers(0, n, e).astype(np.int32) for _ in range(2))
        gs.append((s, d, 0 if g % 5 == 4 else n))
    want = []
    for s, d, n in gs:
        rp, col = gpu.Graph.from_coo(s, d, n or int(max(s.max(initial=0), d.max(initial=0))) + 1).csr()
        want.append(orc.tc_merge(rp, col, threads=1))
    total, per, _ = p.count_batch(gs)
    assert list(per) == want and total == sum(want)
    for bad in (-1, 1500):
        worse = [(s.copy(), d, n) for s, d, n in gs] + [(np.array([0, bad], np.int32), np.array([1, 1], np.int32), 7)]
        worse = worse[-64:]
        with pytest.raises(gpu.BtcError, match="graph %d: vertex id" % (len(worse) - 1)):
            p.count_batch(worse)
        assert list(p.export_batch().count()[1]) == want
    total, per, _ = p.count_batch(gs[::-1])
    assert list(per) == want[::-1]
