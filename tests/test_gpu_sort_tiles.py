"""The captured build with sort tiles of 4096 keys (capacities above 2^20):
pairs, ids and lists of every sort around one and several tiles, on a graph
replayed after runs of other sizes, one graph and several a run; L, labels and
counts equal the host canonicalisation's and the oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TILE = 4096
E_CAP = (1 << 20) + 5


def _pairs(rng, n, e, kind):
    if kind == "random":
        return rng.integers(0, n, e), rng.integers(0, n, e)
    if kind == "star":
        return np.full(e, n - 1), rng.integers(0, n, e)
    return np.full(e, 3 % n), np.full(e, 1 % n)  # one pair, repeated


def _check(orc, p, host, total):
    rp, col = host.csr()
    q = p.graph()
    rp2, col2 = q.csr()
    assert np.array_equal(rp, rp2) and np.array_equal(col, col2)
    assert np.array_equal(host.labels(), q.labels())
    assert total == orc.tc_merge(rp, col, threads=4)


@pytest.mark.parametrize("flags", [0, 2, 3])
def test_pairs_and_ids_around_tiles(gpu, orc, flags):
    p = gpu.Pipeline(1 << 15, E_CAP, flags)
    rng = np.random.default_rng(flags)
    sizes = [E_CAP, 0, 1, 2, TILE - 1, TILE, TILE + 1, 3 * TILE + 7, 40 * TILE]
    ids = [1 << 15, 1, TILE - 1, TILE, TILE + 1, 3 * TILE + 7]
    for k, e in enumerate(sizes + sizes[:0:-1]):
        n = ids[k % len(ids)]
        s, d = (x.astype(np.int32) for x in _pairs(rng, n, e, ("random", "star", "same")[k % 3]))
        total, _ = p.count(s, d, n)
        _check(orc, p, gpu.Graph.from_coo(s, d, n, flags), total)


@pytest.mark.parametrize("k", [1, 5, 64])
def test_several_graphs(gpu, orc, k):
    p = gpu.Pipeline(1 << 17, E_CAP, 3, max_graphs=64)
    rng = np.random.default_rng(k)
    for sizes in ([E_CAP // k] * k, [1] * k, [TILE // k + 1] * k, [3 * TILE // k + 7] * k):
        gs = []
        for e in sizes:
            n = int(rng.integers(2, (1 << 17) // k))
            gs.append(tuple(rng.integers(0, n, e).astype(np.int32) for _ in range(2)) + (n,))
        want = [orc.tc_merge(*gpu.Graph.from_coo(*g).csr(), threads=4) for g in gs]
        total, per, _ = p.count_batch(gs)
        assert list(per) == want and total == sum(want)
        assert list(p.export_batch().count()[1]) == want
