"""Bit-BSR counts of complete and nearly complete graphs: few tiles, nearly all
of them dense, whole row items without a list, and every route of the dense
threshold.  Counts are integers: equality."""
import numpy as np
import pytest

from test_gpu_row_count import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [32, 64, 128])
@pytest.mark.parametrize("n", [300, 513, 530, 1300])
def test_dense_graphs(gpu, orc, n, K):
    u, v = np.triu_indices(n, 1)
    keep = np.random.default_rng(n).random(u.size) < 0.97
    for a, b in ((u, v), (u[keep], v[keep])):
        check(gpu, orc, a.astype(np.int32), b.astype(np.int32), n, K, [-1, 0, 40, 16 * K])
