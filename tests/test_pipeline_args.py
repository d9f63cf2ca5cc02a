"""Pipeline.count_batch refuses what it cannot read before it reaches the
library: no device is needed."""
import numpy as np
import pytest


@pytest.mark.parametrize("graphs,error", [
    ([], ValueError),
    ([(5, 6, 7)], TypeError),
    ([(np.int32(5), np.int32(6), 7)], TypeError),
    ([([0, 1], [1, 2], 3), (np.array(4), [1], 5)], TypeError),
    ([([0, 1], [1], 3)], ValueError),
    ([([0], [1], 3), ([0, 1], [1, 0, 2], 3)], ValueError),
])
def test_count_batch_arguments(btc, graphs, error):
    p = object.__new__(btc.Pipeline)
    p._h = None
    with pytest.raises(error):
        p.count_batch(graphs)
