"""Set bits of a Bit-BSR's tiles around 32, where their copies beside the
entries change hands: thresholds on either side of every tile send each entry
down exactly one path."""
import numpy as np
import pytest

from test_gpu_row_count import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [32, 64, 128])
@pytest.mark.parametrize("n", [250, 1007])
def test_tile_pops(gpu, orc, n, K):
    rng = np.random.default_rng(n + K)
    u, v = np.triu_indices(n, 1)
    # bits a tile: 0 to 80, another share in every 16 x K block
    share = rng.integers(0, 81, (n // 16 + 1, n // K + 1)) / (16 * K)
    keep = rng.random(u.size) < share[v // 16, u // K]
    keep[: n // 2] = True  # one long row and column
    check(gpu, orc, u[keep].astype(np.int32), v[keep].astype(np.int32), n, K, [-1, 0, 1, 30, 31, 32, 33, 60])
