"""Degree order of the GPU canonicalisation on both sides of the rule for its
degree copies (edges per id, few ids), ids without edges included."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,e", [(1, 0), (5, 3), (1 << 17, 1 << 10), ((1 << 17) + 1, 1 << 10),
                                 ((1 << 17) + 1, (1 << 18) + 5), (1 << 18, 1 << 17), (1 << 18, 3 << 18)])
@pytest.mark.parametrize("flags", [2, 3])
def test_degree_order(gpu, n, e, flags):
    rng = np.random.default_rng(n + e)
    s, d = (rng.integers(0, n, e).astype(np.int32) for _ in range(2))
    if e > 1000:  # a hub, and one near the end of the ids
        s[:300], s[300:500] = 7, n - 2
    host = gpu.Graph.from_coo(s, d, n, flags)
    dev = gpu.Graph.from_coo(s, d, n, flags | gpu.CANON_DEVICE)
    for a, b in zip(host.csr(), dev.csr()):
        assert np.array_equal(a, b)
    assert np.array_equal(host.labels(), dev.labels())
