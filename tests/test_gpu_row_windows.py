"""Bit-BSR counts of rows that fit neither LDS set (more than 2048 ids over a
span beyond one bitmap window of 131,040 ids), with ids on the windows' edges
and lists that cross them.  Counts are integers: equality."""
import numpy as np
import pytest

from test_gpu_row_count import check

pytestmark = pytest.mark.gpu

SPAN = 32 * 4095


def wide_rows(lengths, n0, first, seed):
    """Rows n0 + k of lengths[k] ids in [first, n0) each, a third of them from
    a shared pool with the edges of the windows, and all rows below them."""
    rng = np.random.default_rng(seed)
    edges = np.arange(first & ~31, n0, SPAN)[:, None] + np.array([-33, -32, -31, -2, -1, 0, 1, 31, 32])
    pool = np.unique(np.concatenate([edges.ravel(), rng.integers(first, n0, 6000), [first, n0 - 1]]))
    pool = pool[(pool >= first) & (pool < n0)]
    s, d = [rng.choice(pool, 20000)], [rng.choice(pool, 20000)]
    for k, m in enumerate(lengths):
        ids = np.unique(np.concatenate([rng.choice(pool, min(m // 3, pool.size), replace=False),
                                        rng.integers(first, n0, m), [first, n0 - 1]]))
        ids = np.concatenate([ids, n0 + np.arange(k)])
        s.append(np.full(ids.size, n0 + k))
        d.append(ids)
    return np.concatenate(s), np.concatenate(d), n0 + len(lengths)


@pytest.mark.parametrize("K", [32, 128])
@pytest.mark.parametrize("n0,first", [(SPAN + 32, 0), (SPAN + 33, 0), (SPAN + 64, 31), (2 * SPAN, 32),
                                      (2 * SPAN + 1, 0), (400000, 77), (3 * SPAN + 5, 64)])
def test_windows(gpu, orc, n0, first, K):
    lengths = [2040, 2060, 2500, 5000, 12000, 40, 30000, 2100, 300, 9000, 2300] + [2200] * 30
    s, d, n = wide_rows(lengths, n0, first, n0 + first + K)
    check(gpu, orc, s.astype(np.int32), d.astype(np.int32), n, K, [-1, 8, 16 * K])


@pytest.mark.parametrize("K", [32, 128])
def test_more_lists_than_an_item_holds(gpu, orc, K):
    """320 wide rows below one another: items of 256 lists, the last ones long."""
    s, d, n = wide_rows([2100 + 3 * k for k in range(320)], 300000, 5, K)
    check(gpu, orc, s.astype(np.int32), d.astype(np.int32), n, K, [-1, 200])
