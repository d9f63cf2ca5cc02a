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
