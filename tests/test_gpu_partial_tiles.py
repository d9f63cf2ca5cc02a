"""Plans whose own Bit-BSR holds only the row blocks their dense tiles need:
totals, per-vertex counts and the plan's edge split equal those of a plan on
the caller's whole Bit-BSR and the host planner's, for dense tiles in the
first, last and ragged row blocks and for none."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _graph(gpu, kind, n, rng):
    s, d = (rng.integers(0, n, 6 * n) for _ in range(2))
    if kind == "none":
        return s, d
    base = {"first": 0, "last": n - 90, "two": 32}[kind]  # a clique of 90 ids
    x, y = np.triu_indices(90, 1)
    s, d = np.append(s, base + x), np.append(d, base + y)
    if kind == "two":
        s, d = np.append(s, n - 95 + x), np.append(d, n - 95 + y)
    return s, d


@pytest.mark.parametrize("tile_k", [32, 64, 128])
@pytest.mark.parametrize("kind", ["none", "first", "last", "two"])
@pytest.mark.parametrize("n", [200, 3001])
def test_partial_tiles(gpu, orc, n, kind, tile_k):
    rng = np.random.default_rng(n + tile_k)
    s, d = (x.astype(np.int32) for x in _graph(gpu, kind, n, rng))
    g = gpu.Graph.from_coo(s, d, n, gpu.CANON_DEVICE)
    rp, col = g.csr()
    want, rows = orc.tc_merge(rp, col, threads=4, per_row=True)
    for tau in (-1, 0, 20):
        p = gpu.Plan(g, planner=2, tile_k=tile_k, tau=tau)
        total, pv, _ = p.count(per_vertex=True)
        assert total == want and np.array_equal(pv, rows)
        assert p.count()[0] == want
        q = gpu.Plan(g, planner=1, tile_k=tile_k, tau=tau)
        for k in ("dense_tiles", "dense_edges", "sparse_edges"):
            assert p.info[k] == q.info[k], k
        assert q.count()[0] == want
