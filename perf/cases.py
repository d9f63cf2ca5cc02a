"""What the engine's users have it do, as cases that can be timed.

Each case is one call path through the public Python API over the sizes that
the framework is used at: counts of a graph whose plan is resident, the
reference-semantics tile count of a Bit-BSR, whole builds from pairs, the
captured pipeline of new small graphs and batches of many graphs.  Graph
families and sizes are the benchmark's (R-MAT with edge factor 16 and
(0.57, 0.19, 0.19), Erdos-Renyi, 27-point stencils, planted communities, the
serving and batched workloads' size ranges).  Pairs are drawn on the GPU from
the case's seed, so another seed gives another graph.

  listed()          the cases, by name
  draw(rng)         one more case of the same ranges
  prepare(case, s)  the state before the timed call (inputs, graphs, plans)
  run(state)        one pass
  work(case)        bytes and operations one pass cannot do without
  exact(case, s)    the same outputs from a plain wedge enumeration in int64
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "btc-tc-artifact_amd"))

import btc_amd as btc  # noqa: E402

DEV = "cuda"
RMAT = (0.57, 0.19, 0.19)


def listed():
    return [
        # Counts of a resident graph.  The smallest call a user makes in a
        # loop: launches and the copy back decide.
        {"name": "count-er-16k", "path": "count", "family": "er", "n": 16384, "degree": 16.0, "order": "degree",
         "per_vertex": False},
        # A community graph in its natural order, whose dense tiles take the
        # bit-tile kernel.
        {"name": "count-planted-128k", "path": "count", "family": "planted", "n": 1 << 17, "community": 128,
         "p": 0.5, "noise": 4.0, "order": "natural", "per_vertex": False},
        # Local counts: every vertex's triangles of a skewed graph.
        {"name": "count-rmat-18-pv", "path": "count", "family": "rmat", "n": 1 << 18, "degree": 16, "order": "degree",
         "per_vertex": True},
        # The headline graph, resident: bandwidth decides.
        {"name": "count-rmat-22", "path": "count", "family": "rmat", "n": 1 << 22, "degree": 16, "order": "degree",
         "per_vertex": False},
        # The reference's own count calls on a Bit-BSR (drop-in callers of
        # the 16x32 and 16x128 kernels): sparse tiles, dense tiles, hubs.
        {"name": "tiles-er-16k", "path": "tiles", "family": "er", "n": 16384, "degree": 16.0, "tile_k": 32,
         "per_vertex": False, "mfma": False},
        {"name": "tiles-planted-128k", "path": "tiles", "family": "planted", "n": 1 << 17, "community": 128,
         "p": 0.5, "noise": 4.0, "tile_k": 128, "per_vertex": False, "mfma": False},
        {"name": "tiles-rmat-17-pv", "path": "tiles", "family": "rmat", "n": 1 << 17, "degree": 16, "tile_k": 128,
         "per_vertex": True, "mfma": False},
        # The reference's command line from pairs in host memory: canonical
        # form in id order, tiles of the width its rule picks, one count.
        {"name": "lite-stencil-64", "path": "lite", "family": "stencil", "nx": 64, "ny": 64, "nz": 64,
         "per_vertex": False},
        # A new large graph whose pairs are in HBM already, counted once.
        {"name": "oneshot-rmat-20", "path": "oneshot", "family": "rmat", "n": 1 << 20, "degree": 16,
         "per_vertex": False},
        # Serving: a new graph of the stream's median size, and a backlog's
        # group of them, through the captured pipeline from host pairs.
        {"name": "pipeline-rmat-8k", "path": "pipeline", "n": 8192, "degree": 16},
        {"name": "pipeline-group-24", "path": "group", "graphs": 24, "n_lo": 2048, "n_hi": 24576, "degree": 16},
        # Many small graphs of three families, resident, in one launch.
        {"name": "batch-512", "path": "batch", "graphs": 512, "n_lo": 256, "n_hi": 16384},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _family(rng, n_hi):
    f = rng.choice(["er", "rmat", "rmat", "planted", "stencil"])
    if f == "er":
        return {"family": f, "n": _log(rng, 1024, n_hi), "degree": round(rng.uniform(4, 32), 2)}
    if f == "rmat":
        return {"family": f, "n": _log(rng, 1024, n_hi), "degree": rng.randint(8, 16)}
    if f == "planted":
        return {"family": f, "n": _log(rng, 1024, min(n_hi, 1 << 17)), "community": rng.randint(24, 160),
                "p": round(rng.uniform(0.2, 0.7), 3), "noise": round(rng.uniform(0.5, 6), 2)}
    hi = max(16, min(64, int(n_hi ** (1 / 3))))
    return {"family": f, "nx": rng.randint(8, hi), "ny": rng.randint(8, hi), "nz": rng.randint(8, hi)}


def draw(rng):
    path = rng.choice(["count", "count", "tiles", "tiles", "lite", "oneshot", "pipeline", "group", "batch"])
    c = {"path": path}
    if path == "count":
        c.update(_family(rng, 1 << 20))
        c["order"] = rng.choice(["degree", "degree", "natural"])
        c["per_vertex"] = rng.random() < 0.4
        if c["family"] == "rmat" and c["order"] == "natural":  # id-ordered hubs make far longer lists
            c["n"] = min(c["n"], 200000)
    elif path == "tiles":
        c.update(_family(rng, 1 << 17))
        c["tile_k"] = rng.choice([32, 64, 128])
        c["per_vertex"] = rng.random() < 0.4
        c["mfma"] = rng.random() < 0.25
    elif path == "lite":
        c.update(_family(rng, 1 << 17))
        c["per_vertex"] = rng.random() < 0.3
    elif path == "oneshot":
        c.update(_family(rng, 1 << 20))
        c["per_vertex"] = rng.random() < 0.3
    elif path == "pipeline":
        c.update({"n": _log(rng, 64, 1 << 17), "degree": rng.randint(8, 16)})
    elif path == "group":
        lo = _log(rng, 64, 4096)
        c.update({"graphs": rng.randint(2, 64), "n_lo": lo, "n_hi": rng.randint(lo, 16384),
                  "degree": rng.randint(8, 16)})
    else:
        c.update({"graphs": rng.randint(16, 512), "n_lo": 256, "n_hi": _log(rng, 1024, 16384)})
    return c


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)
    return g


def _rmat(n, degree, gen):
    """R-MAT pairs of 2^ceil(log2 n) ids, those with an id >= n dropped."""
    scale = max(1, math.ceil(math.log2(n)))
    a, b, c = RMAT
    k = int(degree) << scale
    u = torch.zeros(k, dtype=torch.int32, device=DEV)
    v = torch.zeros(k, dtype=torch.int32, device=DEV)
    for _ in range(scale):
        r = torch.rand(k, generator=gen, device=DEV)
        u.mul_(2).add_((r >= a + b).int())
        v.mul_(2).add_((((r >= a) & (r < a + b)) | (r >= a + b + c)).int())
    if n < 1 << scale:
        keep = (u < n) & (v < n)
        u, v = u[keep], v[keep]
    return u, v, n


def _er(n, degree, gen):
    k = max(1, int(n * degree / 2))
    uv = torch.randint(0, n, (2, k), generator=gen, device=DEV, dtype=torch.int32)
    return uv[0].contiguous(), uv[1].contiguous(), n


def _planted(n, community, p, noise, gen):
    x, y = torch.triu_indices(community, community, 1, device=DEV)
    first = torch.arange(0, n, community, device=DEV)
    us, vs = [], []
    for part in first.split(256):
        u = (part[:, None] + x[None, :]).reshape(-1)
        v = (part[:, None] + y[None, :]).reshape(-1)
        keep = (torch.rand(u.numel(), generator=gen, device=DEV) < p) & (v < n)
        us.append(u[keep].int())
        vs.append(v[keep].int())
    a, b, _ = _er(n, noise, gen)
    return torch.cat(us + [a]), torch.cat(vs + [b]), n


def _stencil(nx, ny, nz, gen):
    """27-point stencil of a mesh with 2 % of its cells removed."""
    n = nx * ny * nz
    live = torch.rand(nx, ny, nz, generator=gen, device=DEV) >= 0.02
    idx = torch.arange(n, device=DEV, dtype=torch.int32).reshape(nx, ny, nz)
    us, vs = [], []
    for dx in (0, 1):
        for dy in (-1, 0, 1):
            for dz in (-1, 0, 1):
                if (dx, dy, dz) <= (0, 0, 0):
                    continue
                s = tuple(slice(max(0, -d), m - max(0, d)) for d, m in ((dx, nx), (dy, ny), (dz, nz)))
                t = tuple(slice(max(0, d), m - max(0, -d)) for d, m in ((dx, nx), (dy, ny), (dz, nz)))
                keep = live[s] & live[t]
                us.append(idx[s][keep])
                vs.append(idx[t][keep])
    return torch.cat(us), torch.cat(vs), n


def _stencil2d(a, b, gen):
    """9-point stencil of an a x b mesh with 2 % of its cells removed."""
    return _stencil(1, a, b, gen)


def _pairs(case, gen):
    f = case["family"]
    if f == "rmat":
        return _rmat(case["n"], case["degree"], gen)
    if f == "er":
        return _er(case["n"], case["degree"], gen)
    if f == "planted":
        return _planted(case["n"], case["community"], case["p"], case["noise"], gen)
    return _stencil(case["nx"], case["ny"], case["nz"], gen)


def _many(case, seed):
    """The graphs of a group (R-MAT) or of a batch (40 % Erdos-Renyi, 40 %
    R-MAT, 20 % 9-point stencils), n log-uniform in the case's range."""
    rng = np.random.default_rng(seed)
    gen = _gen(seed)
    out = []
    for _ in range(case["graphs"]):
        n = int(round(math.exp(rng.uniform(math.log(case["n_lo"]), math.log(case["n_hi"])))))
        r = rng.random()
        if case["path"] == "group":
            out.append(_rmat(n, case["degree"], gen))
        elif r < 0.4:
            out.append(_er(n, float(rng.uniform(8, 32)), gen))
        elif r < 0.8:
            out.append(_rmat(n, int(rng.integers(8, 17)), gen))
        else:
            a = math.isqrt(n)
            out.append(_stencil2d(a, n // a, gen))
    return out


def _host(g):
    u, v, n = g
    return u.cpu().numpy(), v.cpu().numpy(), n


def _flags(case):
    """Canonical form: degree order for the engine, id order for tiles;
    local counts keep the caller's id space (no compaction)."""
    by_degree = case["path"] == "oneshot" or (case["path"] == "count" and case["order"] == "degree")
    return (btc.CANON_DEGREE_ORDER if by_degree else 0) | (0 if case["per_vertex"] else btc.CANON_COMPACT)


def _cap(x):
    return 1 << max(6, math.ceil(math.log2(max(2, x))))


# ------------------------------------------------------------ state and pass
def prepare(case, seed):
    path = case["path"]
    st = {"path": path, "per_vertex": case.get("per_vertex", False)}
    if path in ("group", "batch"):
        graphs = [_host(g) for g in _many(case, seed)]
        if path == "batch":
            st["batch"] = btc.Batch.from_coo(graphs)
        else:
            st["graphs"] = graphs
            st["pipe"] = btc.Pipeline(_cap(sum(g[2] for g in graphs)), _cap(sum(len(g[0]) for g in graphs)),
                                      max_graphs=max(2, case["graphs"]))
    elif path == "pipeline":
        u, v, n = _host(_rmat(case["n"], case["degree"], _gen(seed)))
        st.update(u=u, v=v, n=n, pipe=btc.Pipeline(_cap(n), _cap(u.size)))
    else:
        u, v, n = _pairs(case, _gen(seed))
        torch.cuda.synchronize()
        if path == "oneshot":
            st.update(u=u, v=v, n=n, flags=_flags(case))
        elif path == "lite":
            st.update(u=u.cpu().numpy(), v=v.cpu().numpy(), n=n, flags=_flags(case) | btc.CANON_DEVICE)
        else:
            g = btc.Graph.from_coo_device(u.data_ptr(), v.data_ptr(), u.numel(), n, _flags(case))
            st["graph"] = g
            if path == "tiles":
                st["tiles"] = btc.BitBSR(g, case["tile_k"])
                st["mfma"] = case["mfma"]
            else:
                st["plan"] = btc.Plan(g)
    return st


def run(st):
    path, pv = st["path"], st["per_vertex"]
    if path == "count":
        total, rows, _ = st["plan"].count(per_vertex=pv)
    elif path == "tiles":
        total, rows, _ = st["tiles"].count(per_vertex=pv, mfma=st["mfma"])
    elif path == "lite":
        g = btc.Graph.from_coo(st["u"], st["v"], st["n"], st["flags"])
        b = btc.BitBSR(g, btc.lite_tile_k(g.n, g.m))
        total, rows, _ = b.count(per_vertex=pv)
        b.close()
        g.close()
    elif path == "oneshot":
        g = btc.Graph.from_coo_device(st["u"].data_ptr(), st["v"].data_ptr(), st["u"].numel(), st["n"], st["flags"])
        p = btc.Plan(g)
        total, rows, _ = p.count(per_vertex=pv)
        p.close()
        g.close()
    elif path == "pipeline":
        total, _ = st["pipe"].count(st["u"], st["v"], st["n"])
        return total
    elif path == "group":
        total, per, _ = st["pipe"].count_batch(st["graphs"])
        return total, per
    else:
        total, per, _ = st["batch"].count()
        return total, per
    return (total, rows) if pv else total


# -------------------------------------------------------------------- sizes
def _size(case):
    """(vertices, pairs) expected of the case's graph."""
    f = case.get("family", "rmat")
    if case["path"] in ("group", "batch"):
        lo, hi = case["n_lo"], max(case["n_lo"] + 1, case["n_hi"])
        mean = (hi - lo) / math.log(hi / lo)
        return case["graphs"] * mean, case["graphs"] * mean * (case["degree"] if case["path"] == "group" else 9.0)
    if f == "stencil":
        n = case["nx"] * case["ny"] * case["nz"]
        return n, 12.5 * n
    n = case["n"]
    if f == "planted":
        return n, n * ((case["community"] - 1) * case["p"] + case["noise"]) / 2
    if f == "er":
        return n, n * case["degree"] / 2
    return n, n * case["degree"]


def work(case):
    """Bytes: the pairs of a path that starts from them, or the canonical L
    (row offsets and columns) of a resident graph, and the results.
    Operations: one membership test per edge of L at the least."""
    n, e = _size(case)
    resident = case["path"] in ("count", "tiles", "batch")
    out = 8 + (4 * n if case.get("per_vertex") else 0) + 8 * case.get("graphs", 0)
    return {"bytes": float((4 * (n + 1) + 4 * e if resident else 8 * e) + out), "flops": float(e)}


# -------------------------------------------------------------------- exact
def _canonical(u, v, n, by_degree, compact=True, seg=None):
    """Sorted keys row << 32 | col of L over n' ids (the used ones when
    compacted), in id order or by descending degree (ties by id), and each
    row's segment."""
    u, v = u.long(), v.long()
    k = torch.unique((torch.maximum(u, v) << 32) | torch.minimum(u, v))
    k = k[(k >> 32) != (k & 0xFFFFFFFF)]
    r, c = k >> 32, k & 0xFFFFFFFF
    deg = torch.bincount(r, minlength=n) + torch.bincount(c, minlength=n)
    ids = torch.nonzero(deg).flatten() if compact else torch.arange(n, device=u.device)
    if by_degree:
        ids = ids[torch.argsort(deg[ids], descending=True, stable=True)]
    rank = torch.zeros(n, dtype=torch.int64, device=u.device)
    rank[ids] = torch.arange(ids.numel(), device=u.device)
    r, c = rank[r], rank[c]
    k = torch.sort((torch.maximum(r, c) << 32) | torch.minimum(r, c))[0]
    return k, ids.numel(), seg[ids] if seg is not None else None


def _row_counts(k, n):
    """Triangles of every row of L: wedges (i; j, k) of row i with (j, k) in L."""
    rows, cols = k >> 32, k & 0xFFFFFFFF
    ptr = torch.searchsorted(rows.contiguous(), torch.arange(n + 1, device=k.device))
    before = torch.arange(k.numel(), device=k.device) - ptr[rows]
    ends = torch.cumsum(before, 0)
    out = torch.zeros(n, dtype=torch.int64, device=k.device)
    step, e0, total = 1 << 25, 0, int(ends[-1]) if k.numel() else 0
    if total > 3_000_000_000:
        return None
    while e0 < k.numel():
        base = int(ends[e0 - 1]) if e0 else 0
        e1 = max(e0 + 1, int(torch.searchsorted(ends, torch.tensor(base + step, device=k.device), right=True)))
        q = torch.repeat_interleave(torch.arange(e0, e1, device=k.device), before[e0:e1])
        if q.numel():
            off = torch.arange(q.numel(), device=k.device) - (ends[q] - before[q] - base)
            want = (cols[q] << 32) | cols[ptr[rows[q]] + off]
            at = torch.searchsorted(k, want).clamp_(max=k.numel() - 1)
            out += torch.bincount(rows[q][k[at] == want], minlength=n)
        e0 = e1
    return out


def exact(case, seed):
    path = case["path"]
    if path in ("group", "batch"):
        us, vs, segs, n0 = [], [], [], 0
        for j, (u, v, n) in enumerate(_many(case, seed)):
            us.append(u.long() + n0)
            vs.append(v.long() + n0)
            segs.append(torch.full((n,), j, dtype=torch.int64, device=DEV))
            n0 += n
        k, nc, seg = _canonical(torch.cat(us), torch.cat(vs), n0, True, seg=torch.cat(segs))
        rows = _row_counts(k, nc)
        if rows is None:
            return None
        per = torch.zeros(case["graphs"], dtype=torch.int64, device=DEV).index_add_(0, seg, rows)
        return int(per.sum()), per.cpu().numpy().astype(np.uint64)
    if path == "pipeline":
        u, v, n = _rmat(case["n"], case["degree"], _gen(seed))
        flags = btc.CANON_DEFAULT
    else:
        u, v, n = _pairs(case, _gen(seed))
        flags = _flags(case)
    k, nc, _ = _canonical(u, v, n, bool(flags & btc.CANON_DEGREE_ORDER), bool(flags & btc.CANON_COMPACT))
    rows = _row_counts(k, nc)
    if rows is None:
        return None
    total = int(rows.sum())
    return (total, rows.cpu().numpy().astype(np.int32)) if case.get("per_vertex") else total
