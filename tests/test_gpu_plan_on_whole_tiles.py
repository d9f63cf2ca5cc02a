"""Plans whose own Bit-BSR holds only the row blocks their dense tiles need
against plans on the caller's whole Bit-BSR of the same graph: totals, every
vertex's count and the plan's split."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_partial_tiles import _graph

pytestmark = pytest.mark.gpu


def _plan_on(gpu, b, g, **opts):
    """btc_plan_create_on_bitbsr as a Plan."""
    p = gpu.Plan.__new__(gpu.Plan)
    p.graph, p.opts, p.tiles = g, gpu.make_opts(**opts), b
    p._h = C.c_void_p()
    fn = gpu.lib().btc_plan_create_on_bitbsr
    fn.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.POINTER(C.c_void_p)]
    assert fn(g._h, b._h, C.byref(p.opts), None, C.byref(p._h)) == 0, gpu.lib().btc_last_error()
    return p


@pytest.mark.parametrize("tile_k", [32, 64, 128])
@pytest.mark.parametrize("kind", ["none", "first", "last", "two"])
def test_same_as_on_whole_tiles(gpu, orc, kind, tile_k):
    n = 3001
    s, d = (x.astype(np.int32) for x in _graph(gpu, kind, n, np.random.default_rng(tile_k)))
    g = gpu.Graph.from_coo(s, d, n, gpu.CANON_DEVICE)
    want, rows = orc.tc_merge(*g.csr(), threads=4, per_row=True)
    b = gpu.BitBSR(g, tile_k)
    for tau in (-1, 0, 20):
        for planner in (1, 2):
            own = gpu.Plan(g, planner=planner, tile_k=tile_k, tau=tau)
            ext = _plan_on(gpu, b, g, planner=planner, tile_k=tile_k, tau=tau)
            for p in (own, ext):
                total, pv, _ = p.count(per_vertex=True)
                assert total == want and np.array_equal(pv, rows)
                assert p.count()[0] == want
            for k in ("dense_tiles", "dense_edges", "sparse_edges", "work_items", "wedge_checks"):
                assert own.info[k] == ext.info[k], k
            own.close()
            ext.close()
