"""Calls that still fit when the device is nearly full: a GPU-planned plan in
the bytes that lists, keys and prefix sums of every entry take (60 a list), and
an explicit small threshold whose dense units find no room."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MIB = 1 << 20


class Fill:
    """Allocates device memory until `leave` bytes are free."""

    def __init__(self):
        self.hip = C.CDLL("libamdhip64.so")
        self.hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
        self.hip.hipFree.argtypes = [C.c_void_p]
        self.held = []

    def free(self):
        a, b = C.c_size_t(), C.c_size_t()
        assert self.hip.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    def leave(self, nbytes):
        while True:
            size = min(self.free() - nbytes, 32 << 30) // (2 * MIB) * 2 * MIB
            if size <= 0:
                return
            p = C.c_void_p()
            assert self.hip.hipMalloc(C.byref(p), size) == 0
            self.held.append(p)

    def drop(self):
        while self.held:
            assert self.hip.hipFree(self.held.pop()) == 0


def max_lists(rp, col):
    """Entries whose prefix may meet the pivot's id range."""
    n = rp.size - 1
    row = np.repeat(np.arange(n), np.diff(rp))
    q = np.arange(col.size)
    has = np.diff(rp) > 0
    lo, hi = np.zeros(n, np.int64), np.full(n, -1, np.int64)
    lo[has] = col[rp[:-1][has]]
    hi[has] = col[rp[1:][has] - 1]
    first = rp[row]
    return int(np.count_nonzero((q > first) & (col[np.maximum(q - 1, 0)] >= lo[col]) & (col[first] <= hi[col])))


def test_nearly_full_device(gpu, orc):
    s, d = gpu.gen_rmat(20, 16, seed=3)
    g = gpu.Graph.from_coo(s, d, 1 << 20, gpu.CANON_DEFAULT | gpu.CANON_DEVICE)
    rp, col = g.csr()
    want = orc.tc_merge(rp, col, threads=8)
    p = gpu.Plan(g, planner=2, tau=64 * 16)  # no dense tiles
    i = p.info
    p.close()
    b = gpu.BitBSR(g, 32)
    assert b.count(tau=0)[0] == want  # every kernel is loaded by now
    gpu.memory_trim()
    need = 60 * max_lists(rp, col) + i["core_rows"] * i["core_ids"] // 8 + 40 * g.n + 128 * i["work_items"]
    fill = Fill()
    try:
        fill.leave(need + 48 * MIB)
        p = gpu.Plan(g, planner=2, tau=64 * 16)
        assert p.info == i and p.count()[0] == want
        p.close()
        gpu.memory_trim()
        fill.leave(128 * MIB)  # of 500 for 32 bytes a unit
        total, pv, _ = b.count(tau=0, per_vertex=True)
        assert total == want and int(pv.sum()) == want
        assert b.count()[0] == want
    finally:
        fill.drop()
    assert b.count(tau=0)[0] == want
    b.close()
    g.close()
