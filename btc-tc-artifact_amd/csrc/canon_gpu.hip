// Device canonicalisation: COO pairs in HBM -> strictly lower triangle L
// (CSR) in HBM, equal bit for bit to the host path (canon.cpp).
//
// Same steps as btc/operations/convert.h: orient (u, v) to (max, min) and
// drop self-loops (symmetrize_and_triangular_gpu, :281-324), sort and
// deduplicate, compact the used ids in order (remap_node_ids_gpu,
// :387-425); then the optional relabel by descending degree (ties by id).
// A pair is one key row << b | col (b = bits of n), radix-sorted on 2b
// bits; duplicates are dropped by a flag scan; CSR rows are found by a
// binary search of each row's first key.  The host copies of the CSR are
// made only when a host consumer asks (ensure_host).
#include <climits>

#include "devtile.h"
#include "internal.h"

namespace btcx {
namespace {

constexpr int kT = 256;
constexpr unsigned kRedBlocks = 1024;    // eager reductions
constexpr unsigned kCapRedBlocks = 256;  // capacity-sized reductions: about one per CU

int id_bits(int64_t n) {
    int b = 1;
    while (b < 31 && (1ll << b) < n) ++b;
    return b;
}

unsigned grid_for(int64_t n) {
    const int64_t g = (n + kT - 1) / kT;
    return (unsigned)std::max<int64_t>(1, std::min<int64_t>(g, 65536));
}

__global__ void id_range_kernel(const int32_t* __restrict__ src, const int32_t* __restrict__ dst, Cnt nnz_,
                                int32_t* __restrict__ lohi) {
    __shared__ int32_t s_lo[kT / 64], s_hi[kT / 64];
    const int64_t nnz = nnz_.get();
    int32_t lo = INT_MAX, hi = -1;
    for (int64_t e = blockIdx.x * (int64_t)kT + threadIdx.x; e < nnz; e += (int64_t)gridDim.x * kT) {
        const int32_t u = src[e], v = dst[e];
        lo = min(lo, min(u, v));
        hi = max(hi, max(u, v));
    }
    for (int o = 32; o > 0; o >>= 1) {
        lo = min(lo, __shfl_xor(lo, o));
        hi = max(hi, __shfl_xor(hi, o));
    }
    if ((threadIdx.x & 63) == 0) {
        s_lo[threadIdx.x >> 6] = lo;
        s_hi[threadIdx.x >> 6] = hi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kT / 64; ++w) {
            lo = min(lo, s_lo[w]);
            hi = max(hi, s_hi[w]);
        }
        if (lo != INT_MAX) atomicMin(&lohi[0], lo);
        if (hi != -1) atomicMax(&lohi[1], hi);
    }
}

// (u, v) -> (max << b) | min; self-loops become the sentinel (all 2b bits
// set, which no oriented pair reaches since max > min).
__global__ void orient_kernel(const int32_t* __restrict__ src, const int32_t* __restrict__ dst, int64_t nnz, int b,
                              uint64_t sentinel, uint64_t* __restrict__ keys) {
    for (int64_t e = blockIdx.x * (int64_t)kT + threadIdx.x; e < nnz; e += (int64_t)gridDim.x * kT) {
        const uint32_t u = (uint32_t)src[e], v = (uint32_t)dst[e];
        keys[e] = u == v ? sentinel : ((uint64_t)max(u, v) << b) | (uint64_t)min(u, v);
    }
}

// flag[e] = key e is the first of its run and not the sentinel
__global__ void first_flag_kernel(const uint64_t* __restrict__ keys, Cnt n_, uint64_t sentinel,
                                  uint32_t* __restrict__ flag) {
    const int64_t n = n_.get();
    for (int64_t e = blockIdx.x * (int64_t)kT + threadIdx.x; e < n; e += (int64_t)gridDim.x * kT) {
        const uint64_t k = keys[e];
        flag[e] = (k != sentinel && (e == 0 || keys[e - 1] != k)) ? 1u : 0u;
    }
}

__global__ void compact_kernel(const uint64_t* __restrict__ keys, const uint32_t* __restrict__ flag,
                               const uint32_t* __restrict__ pos, Cnt n_, uint64_t* __restrict__ out) {
    const int64_t n = n_.get();
    for (int64_t e = blockIdx.x * (int64_t)kT + threadIdx.x; e < n; e += (int64_t)gridDim.x * kT)
        if (flag[e]) out[pos[e]] = keys[e];
}

__global__ void mark_used_kernel(const uint64_t* __restrict__ keys, Cnt m_, int b, uint32_t* __restrict__ used) {
    const int64_t m = m_.get();
    const uint64_t mask = (1ull << b) - 1;
    for (int64_t e = blockIdx.x * (int64_t)kT + threadIdx.x; e < m; e += (int64_t)gridDim.x * kT) {
        const uint64_t k = keys[e];
        used[k >> b] = 1u;
        used[k & mask] = 1u;
    }
}

// labels[newid[v]] = v for every used v (newid = exclusive scan of used)
__global__ void labels_kernel(const uint32_t* __restrict__ used, const uint32_t* __restrict__ newid, Cnt n_,
                              int32_t* __restrict__ labels) {
    const int64_t n = n_.get();
    for (int64_t v = blockIdx.x * (int64_t)kT + threadIdx.x; v < n; v += (int64_t)gridDim.x * kT)
        if (used[v]) labels[newid[v]] = (int32_t)v;
}

__global__ void iota_kernel(int32_t* __restrict__ x, Cnt n_) {
    const int64_t n = n_.get();
    for (int64_t v = blockIdx.x * (int64_t)kT + threadIdx.x; v < n; v += (int64_t)gridDim.x * kT) x[v] = (int32_t)v;
}

// Rewrites keys (row << b | col) through map (NULL = identity) into
// max(map row, map col) << bn | min(...).
__global__ void relabel_kernel(uint64_t* __restrict__ keys, Cnt m_, int b, const uint32_t* __restrict__ map,
                               int bn) {
    const int64_t m = m_.get();
    const uint64_t mask = (1ull << b) - 1;
    for (int64_t e = blockIdx.x * (int64_t)kT + threadIdx.x; e < m; e += (int64_t)gridDim.x * kT) {
        const uint64_t k = keys[e];
        uint32_t r = (uint32_t)(k >> b), c = (uint32_t)(k & mask);
        if (map) {
            r = map[r];
            c = map[c];
        }
        keys[e] = ((uint64_t)max(r, c) << bn) | (uint64_t)min(r, c);
    }
}

// deg[v] += entries of v in the ascending keys [0, m) (row r = k >> b,
// column c = k & mask).  Rows come in runs, so a wave adds each run of its
// 64 keys with one atomic; columns of ids below kDegWindow (where hub
// vertices of skewed graphs concentrate) are counted in LDS first, so a hub
// gets one global atomic per workgroup rather than one per edge.  The sums
// are kept in kDegCopies copies (`stride` words apart), one per XCD as
// workgroups are dealt to them in turn, since a line that eight L2 caches
// want moves between them.  Bound: the L2's atomic rate on scattered words
// (some 19 G/s).  One copy and one run of 64 keys at a time against this:
// R-MAT 2^20 (14 M edges) 873 -> 541 us, 24 graphs (3.3 M) 280 -> 159 us.
constexpr uint32_t kDegWindow = 8192;
// The eager build keeps the copies from one edge per id on, or for few ids:
// clearing and summing them is 64 bytes of traffic an id.  Builds in degree
// order with 8 copies against one: Erdos-Renyi 2^22 ids with m / n = 1/4, 1/2,
// 1, 2 901 / 1044 / 1379 / 1993 us against 858 / 996 / 1326 / 1947, R-MAT 2^22
// 920 / 1067 / 1428 / 2087 against 922 / 1103 / 1502 / 2304, 2^17 ids and
// fewer 5 to 10 us less whatever the edges.
constexpr int64_t kDegCopyIds = int64_t(1) << 17;

// key_at(e): key e, e < m; every thread of the workgroup calls it with its
// own window h and degree copy.
constexpr int kDegPer = 4;  // runs of 64 keys a wave loads together
template <class KeyAt>
__device__ __forceinline__ void count_degrees(KeyAt&& key_at, int64_t m, int b, uint32_t* h, uint32_t* deg) {
    for (uint32_t i = threadIdx.x; i < kDegWindow; i += kT) h[i] = 0;
    __syncthreads();
    const uint64_t mask = (1ull << b) - 1;
    const uint32_t lane = threadIdx.x & 63;
    for (int64_t base = (blockIdx.x * (int64_t)kT + (threadIdx.x & ~63u)) * kDegPer; base < m;
         base += (int64_t)gridDim.x * kT * kDegPer) {
        uint64_t key[kDegPer];
#pragma unroll
        for (int x = 0; x < kDegPer; ++x) {
            const int64_t e = base + x * 64 + lane;
            key[x] = e < m ? key_at(e) : ~0ull;
        }
#pragma unroll
        for (int x = 0; x < kDegPer; ++x) {
            const bool ok = base + x * 64 + lane < m;
            const uint32_t r = (uint32_t)(key[x] >> b);
            const uint32_t prev = __shfl_up(r, 1);
            const uint64_t starts = __ballot(lane == 0 || prev != r);
            // a run's first lane adds its length: up to the next run, the
            // last key or the wave's end
            const uint64_t ends = (starts | __ballot(!ok)) >> lane >> 1;
            if (ok) {
                if (starts >> lane & 1) {
                    const uint32_t cnt = ends ? (uint32_t)__builtin_ctzll(ends) + 1u : 64u - lane;
                    if (r < kDegWindow) atomicAdd(&h[r], cnt);
                    else atomicAdd(&deg[r], cnt);
                }
                const uint32_t c = (uint32_t)(key[x] & mask);
                if (c < kDegWindow) atomicAdd(&h[c], 1u);
                else atomicAdd(&deg[c], 1u);
            }
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < kDegWindow; i += kT)
        if (h[i]) atomicAdd(&deg[i], h[i]);
}

__global__ __launch_bounds__(kT) void degree_kernel(const uint64_t* __restrict__ keys, int64_t m, int b,
                                                    uint32_t* __restrict__ deg, size_t stride_deg,
                                                    uint32_t copies) {
    __shared__ uint32_t h[kDegWindow];
    count_degrees([&](int64_t e) { return keys[e]; }, m, b, h, deg + (blockIdx.x % copies) * stride_deg);
}

// key = top - degree (ascending = descending degree; top is at least the
// largest degree), value = vertex
__global__ void rank_keys_kernel(const uint32_t* __restrict__ deg, size_t stride_deg, uint32_t copies, Cnt n_,
                                 uint32_t top, uint32_t* __restrict__ key, uint32_t* __restrict__ val) {
    const int64_t n = n_.get();
    for (int64_t v = blockIdx.x * (int64_t)kT + threadIdx.x; v < n; v += (int64_t)gridDim.x * kT) {
        uint32_t d = 0;
        for (uint32_t k = 0; k < copies; ++k) d += deg[k * stride_deg + (size_t)v];
        key[v] = top - d;
        val[v] = (uint32_t)v;
    }
}

// key[r] = segment of vertex order[r] (seg = nseg + 1 ascending vertex
// offsets; the last segment whose start is <= the vertex), val[r] = order[r]
__global__ void segment_keys_kernel(const uint32_t* __restrict__ order, int32_t n, const uint32_t* __restrict__ seg,
                                    int nseg, uint32_t* __restrict__ key, uint32_t* __restrict__ val) {
    for (int64_t r = blockIdx.x * (int64_t)kT + threadIdx.x; r < n; r += (int64_t)gridDim.x * kT) {
        const uint32_t v = order[r];
        int lo = 0, hi = nseg;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (seg[mid] <= v) lo = mid;
            else hi = mid;
        }
        key[r] = (uint32_t)lo;
        val[r] = v;
    }
}

// out[k] = map[at[k]] for k <= nseg (compacted segment starts)
__global__ void gather_kernel(const uint32_t* __restrict__ map, const uint32_t* __restrict__ at, int cnt,
                              uint32_t* __restrict__ out) {
    const int k = blockIdx.x * kT + threadIdx.x;
    if (k < cnt) out[k] = map[at[k]];
}

// rank[order[r]] = r; labels_out[r] = labels_in[order[r]]
__global__ void rank_scatter_kernel(const uint32_t* __restrict__ order, Cnt n_, uint32_t* __restrict__ rank,
                                    const int32_t* __restrict__ labels_in, int32_t* __restrict__ labels_out) {
    const int64_t n = n_.get();
    for (int64_t r = blockIdx.x * (int64_t)kT + threadIdx.x; r < n; r += (int64_t)gridDim.x * kT) {
        const uint32_t v = order[r];
        rank[v] = (uint32_t)r;
        labels_out[r] = labels_in[v];
    }
}

// L from the ascending keys: rowptr[r] = first e with keys[e] >= r << b
// (r = 0..n), col[e] = the key's low b bits, col[m, m + kColPad) = 0; col16
// (when set) gets the low 16 bits of col over the same m + kColPad entries,
// erow (when set) every entry's row.
__global__ void csr_kernel(const uint64_t* __restrict__ keys, Cnt m_, int b, Cnt n_, uint32_t* __restrict__ rowptr,
                           int32_t* __restrict__ col, uint16_t* __restrict__ col16, uint32_t* __restrict__ erow) {
    const int64_t m = m_.get();
    const int64_t n = n_.get();
    const uint64_t mask = (1ull << b) - 1;
    const int64_t stride = (int64_t)gridDim.x * kT;
    const int64_t t0 = blockIdx.x * (int64_t)kT + threadIdx.x;
    for (int64_t r = t0; r <= n; r += stride) {
        const uint64_t t = (uint64_t)r << b;
        int64_t lo = 0, hi = m;
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if (keys[mid] < t) lo = mid + 1;
            else hi = mid;
        }
        rowptr[r] = (uint32_t)lo;
    }
    for (int64_t e = t0; e < m + (int64_t)kColPad; e += stride) {
        const uint64_t k = e < m ? keys[e] : 0;
        const int32_t c = (int32_t)(k & mask);
        col[e] = c;
        if (col16) col16[e] = (uint16_t)c;
        if (erow && e < m) erow[e] = (uint32_t)(k >> b);
    }
}

// out: [0] longest row, [1] sum C(d, 2), [2] sum over edges of d(i) + d(j)
// (rows [0, n), edges [0, m) of L; one atomic per workgroup and word)
__global__ __launch_bounds__(kT) void stats_kernel(const uint32_t* __restrict__ rowptr,
                                                   const int32_t* __restrict__ col, Cnt n_, Cnt m_,
                                                   unsigned long long* __restrict__ out) {
    __shared__ uint64_t lds[kT / 64];
    const int64_t n = n_.get();
    const int64_t m = m_.get();
    const int64_t stride = (int64_t)gridDim.x * kT;
    uint32_t mx = 0;
    uint64_t w = 0, work = 0;
    for (int64_t i = blockIdx.x * (int64_t)kT + threadIdx.x; i < n; i += stride) {
        const uint64_t d = rowptr[i + 1] - rowptr[i];
        mx = max(mx, (uint32_t)d);
        w += d * (d - (d > 0)) / 2;
        work += d * d;
    }
    for (int64_t e = blockIdx.x * (int64_t)kT + threadIdx.x; e < m; e += stride) {
        const int32_t j = col[e];
        work += rowptr[j + 1] - rowptr[j];
    }
    for (int o = 32; o > 0; o >>= 1) mx = max(mx, (uint32_t)__shfl_xor((int)mx, o));
    __shared__ uint32_t s_mx[kT / 64];
    if ((threadIdx.x & 63) == 0) s_mx[threadIdx.x >> 6] = mx;
    w = block_sum_u64<kT>(w, lds);
    work = block_sum_u64<kT>(work, lds);
    if (threadIdx.x == 0) {
        for (int k = 1; k < kT / 64; ++k) mx = max(mx, s_mx[k]);
        if (mx) atomicMax(&out[0], (unsigned long long)mx);
        if (w) atomicAdd(&out[1], (unsigned long long)w);
        if (work) atomicAdd(&out[2], (unsigned long long)work);
    }
}

// ------------------------------------------------- capturable form kernels
// First kernel of a run: clears the run's words (keeping the ones the host
// wrote), the sorts' and scans' words and the graphs' sums.
__global__ __launch_bounds__(kT) void pipe_begin_kernel(PipeCtl* __restrict__ c, uint32_t* __restrict__ seq,
                                                        uint64_t seq_words, unsigned long long* __restrict__ work,
                                                        unsigned long long* __restrict__ per_graph,
                                                        uint32_t max_graphs) {
    const uint64_t t = blockIdx.x * (uint64_t)kT + threadIdx.x, stride = (uint64_t)gridDim.x * kT;
    for (uint64_t i = t; i < seq_words; i += stride)
        if (i != kSeqErr) seq[i] = 0;
    if (per_graph)
        for (uint64_t g = t; g < max_graphs; g += stride) per_graph[g] = 0;
    if (blockIdx.x != 0) return;
    constexpr uint32_t kWords = sizeof(PipeCtl) / 4;
    uint32_t* w = reinterpret_cast<uint32_t*>(c);
    for (uint32_t i = threadIdx.x + kPipeHostWords; i < kWords; i += kT) w[i] = 0;
    __syncthreads();
    if (threadIdx.x == 0) {
        c->lo = INT_MAX;
        c->hi = -1;
        work[0] = 0;  // the count's total and cursors
        work[1] = 0;
    }
}

// The oriented keys of unchecked pairs (ids that no vertex count admits
// become the sentinel: the run is refused then, but its kernels stay in
// bounds), the id range and the sort's digits, in one read of the pairs.
__global__ __launch_bounds__(kT) void orient_checked_kernel(const int32_t* __restrict__ src,
                                                            const int32_t* __restrict__ dst, PipeCtl* __restrict__ c,
                                                            int32_t n_cap, int b, uint64_t sentinel,
                                                            uint64_t* __restrict__ keys, SortUse u) {
    __shared__ DigitHist h;
    __shared__ int32_t s_lo[kT / 64], s_hi[kT / 64];
    const uint32_t nnz = c->nnz, limit = (uint32_t)(c->n_in > 0 ? min(c->n_in, n_cap) : n_cap);
    sort_status_clear(u, nnz);
    int32_t lo = INT_MAX, hi = -1;
    hist_clear(h, u.passes);
    auto one = [&](int32_t x, int32_t y) {
        lo = min(lo, min(x, y));
        hi = max(hi, max(x, y));
        const uint32_t a = (uint32_t)x, e = (uint32_t)y;
        const uint64_t k = (a == e || a >= limit || e >= limit) ? sentinel : ((uint64_t)max(a, e) << b) | min(a, e);
        hist_add(h, u.passes, k);
        return k;
    };
    const uint32_t quads = nnz / 4;  // the arrays are 256-byte aligned
    for (uint64_t q = blockIdx.x * (uint64_t)kT + threadIdx.x; q < quads; q += (uint64_t)gridDim.x * kT) {
        const int4 a = reinterpret_cast<const int4*>(src)[q], e = reinterpret_cast<const int4*>(dst)[q];
        const ulonglong2 k0 = make_ulonglong2(one(a.x, e.x), one(a.y, e.y));
        const ulonglong2 k1 = make_ulonglong2(one(a.z, e.z), one(a.w, e.w));
        reinterpret_cast<ulonglong2*>(keys)[2 * q] = k0;
        reinterpret_cast<ulonglong2*>(keys)[2 * q + 1] = k1;
    }
    if (blockIdx.x == 0 && threadIdx.x < (nnz & 3u)) {
        const uint32_t e = 4 * quads + threadIdx.x;
        keys[e] = one(src[e], dst[e]);
    }
    hist_flush(h, u);
    for (int o = 32; o > 0; o >>= 1) {
        lo = min(lo, __shfl_xor(lo, o));
        hi = max(hi, __shfl_xor(hi, o));
    }
    if ((threadIdx.x & 63) == 0) {
        s_lo[threadIdx.x >> 6] = lo;
        s_hi[threadIdx.x >> 6] = hi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kT / 64; ++w) {
            lo = min(lo, s_lo[w]);
            hi = max(hi, s_hi[w]);
        }
        if (lo != INT_MAX) {
            atomicMin(&c->lo, lo);
            atomicMax(&c->hi, hi);
        }
    }
}

// The first of every run of equal sorted keys (the sentinel apart) to out,
// in order; m = their number; with used set, used[v] = 1 for their ids.
// Workgroup 0 also resolves n (the given count, or the largest id + 1) and
// the refusal bits.
template <int PER>
__global__ __launch_bounds__(kT) void unique_kernel(const uint64_t* __restrict__ keys, PipeCtl* __restrict__ c,
                                                    int32_t n_cap, int b, uint64_t sentinel,
                                                    uint64_t* __restrict__ out, uint32_t* __restrict__ used,
                                                    ScanUse u) {
    __shared__ uint32_t lds[4 * PER + 2];
    __shared__ uint32_t s_tile;
    const uint32_t nnz = c->nnz;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const int32_t lo = nnz ? c->lo : 0, hi = c->hi;
        int64_t nn = c->n_in > 0 ? (int64_t)c->n_in : (int64_t)hi + 1;
        uint32_t st = 0;
        if (lo < 0) st |= kPipeNegativeId;
        if (hi >= nn) st |= kPipeIdRange;
        if (nn > n_cap) {
            st |= kPipeTooManyIds;
            nn = n_cap;
        }
        c->n = (uint32_t)nn;
        c->status = st;
    }
    constexpr uint32_t kTile = kT * PER;
    const uint32_t nt = (uint32_t)(((uint64_t)nnz + kTile - 1) / kTile);
    const uint64_t mask = (1ull << b) - 1;
    for (TileLoop l(u.ticket, nt, &s_tile); l.next();) {
        uint64_t k[PER];
        uint32_t f[PER], pos[PER];
#pragma unroll
        for (int x = 0; x < PER; ++x) {
            const uint64_t e = (uint64_t)l.t * kTile + x * kT + threadIdx.x;
            k[x] = e < nnz ? keys[e] : sentinel;
            f[x] = k[x] != sentinel && (e == 0 || keys[e - 1] != k[x]);
        }
        const uint64_t tot = tile_offsets<uint32_t, PER>(f, pos, lds, u, l.t);
        if (l.t == nt - 1 && threadIdx.x == 0) c->m = (uint32_t)tot;
#pragma unroll
        for (int x = 0; x < PER; ++x)
            if (f[x]) {
                out[pos[x]] = k[x];
                if (used) {
                    used[k[x] >> b] = 1u;
                    used[k[x] & mask] = 1u;
                }
            }
    }
}

// The used ids in order: newid = exclusive scan of used, labels[newid[v]] =
// v, nc = their number; used is left cleared for the next run.  With no edge
// nothing is compacted (labels = identity, nc = n), as in
// canonicalise_device.
template <int PER>
__global__ __launch_bounds__(kT) void newid_kernel(uint32_t* __restrict__ used, PipeCtl* __restrict__ c,
                                                   uint32_t* __restrict__ newid, int32_t* __restrict__ labels,
                                                   ScanUse u) {
    __shared__ uint32_t lds[4 * PER + 2];
    __shared__ uint32_t s_tile;
    const uint32_t n = c->n;
    const bool none = c->m == 0;
    constexpr uint32_t kTile = kT * PER;
    const uint32_t nt = (uint32_t)(((uint64_t)n + kTile - 1) / kTile);
    for (TileLoop l(u.ticket, nt, &s_tile); l.next();) {
        uint32_t f[PER], pos[PER];
#pragma unroll
        for (int x = 0; x < PER; ++x) {
            const uint64_t v = (uint64_t)l.t * kTile + x * kT + threadIdx.x;
            f[x] = 0;
            if (v < n) {
                f[x] = used[v];
                if (f[x]) used[v] = 0;
            }
        }
        const uint64_t tot = tile_offsets<uint32_t, PER>(f, pos, lds, u, l.t);
        if (l.t == nt - 1 && threadIdx.x == 0) {
            newid[n] = (uint32_t)tot;
            c->nc = none ? n : (uint32_t)tot;
        }
#pragma unroll
        for (int x = 0; x < PER; ++x) {
            const uint64_t v = (uint64_t)l.t * kTile + x * kT + threadIdx.x;
            if (v < n) newid[v] = pos[x];
            if (f[x]) labels[pos[x]] = (int32_t)v;
            else if (none && v < n) labels[v] = (int32_t)v;
        }
    }
}

// Between the ids' compaction and the relabel: keys rewritten through newid
// (monotone, so they stay sorted; NULL: no compaction, labels = identity and
// nc = n), the graphs' first vertices of L (csegs), and with deg set the
// degrees, as degree_kernel.
__global__ __launch_bounds__(kT) void pipe_rekey_kernel(uint64_t* __restrict__ keys, PipeCtl* __restrict__ c, int b,
                                                        const uint32_t* __restrict__ newid,
                                                        int32_t* __restrict__ labels,
                                                        const uint32_t* __restrict__ segs,
                                                        uint32_t* __restrict__ csegs, uint32_t* __restrict__ deg,
                                                        size_t stride_deg) {
    __shared__ uint32_t h[kDegWindow];
    const int64_t m = c->m, n = c->n;
    if (csegs && blockIdx.x == 0)
        for (uint32_t g = threadIdx.x; g <= c->graphs; g += kT) csegs[g] = newid && m ? newid[segs[g]] : segs[g];
    if (!newid) {
        const int64_t t0 = blockIdx.x * (int64_t)kT + threadIdx.x;
        for (int64_t v = t0; v < n; v += (int64_t)gridDim.x * kT) labels[v] = (int32_t)v;
        if (t0 == 0) c->nc = (uint32_t)n;
    }
    const uint64_t mask = (1ull << b) - 1;
    auto rekey = [&](int64_t e) -> uint64_t {
        const uint64_t k = keys[e];
        if (!newid) return k;
        const uint64_t x = ((uint64_t)newid[k >> b] << b) | (uint64_t)newid[k & mask];
        keys[e] = x;
        return x;
    };
    if (!deg) {
        if (newid)
            for (int64_t e = blockIdx.x * (int64_t)kT + threadIdx.x; e < m; e += (int64_t)gridDim.x * kT) rekey(e);
        return;
    }
    if (blockIdx.x * (int64_t)kT * kDegPer >= m) return;  // workgroup-uniform: no keys of its own
    count_degrees(rekey, m, b, h, deg + (blockIdx.x % kDegCopies) * stride_deg);
}

// rank_keys_kernel within graphs (csegs set): key = graph << b | (top -
// degree), so one sort orders by (graph, descending degree, id).  The degree
// copies are left cleared for the next run; the sort's digits are taken.
__global__ __launch_bounds__(kT) void pipe_rank_keys_kernel(uint32_t* __restrict__ deg, size_t stride_deg,
                                                            const PipeCtl* __restrict__ c,
                                                            const uint32_t* __restrict__ csegs, uint32_t top, int b,
                                                            uint32_t* __restrict__ key, uint32_t* __restrict__ val,
                                                            SortUse u) {
    __shared__ DigitHist h;
    const int64_t n = c->nc;
    sort_status_clear(u, (uint64_t)n);
    hist_clear(h, u.passes);
    for (int64_t v = blockIdx.x * (int64_t)kT + threadIdx.x; v < n; v += (int64_t)gridDim.x * kT) {
        uint32_t lo = 0;
        if (csegs) {
            uint32_t hi = c->graphs;  // the last graph whose first vertex is <= v
            while (hi - lo > 1) {
                const uint32_t mid = (lo + hi) >> 1;
                if (csegs[mid] <= (uint32_t)v) lo = mid;
                else hi = mid;
            }
        }
        uint32_t part[kDegCopies], d = 0;
#pragma unroll
        for (uint32_t k = 0; k < kDegCopies; ++k) part[k] = deg[k * stride_deg + (size_t)v];
#pragma unroll
        for (uint32_t k = 0; k < kDegCopies; ++k) {
            d += part[k];
            if (part[k]) deg[k * stride_deg + (size_t)v] = 0;
        }
        const uint32_t x = (csegs ? lo << b : 0u) | (top - d);
        key[v] = x;
        val[v] = (uint32_t)v;
        hist_add(h, u.passes, x);
    }
    hist_flush(h, u);
}

// relabel_kernel through rank, with the next sort's digits.
__global__ __launch_bounds__(kT) void pipe_relabel_kernel(uint64_t* __restrict__ keys, const PipeCtl* __restrict__ c,
                                                          int b, const uint32_t* __restrict__ rank, SortUse u) {
    __shared__ DigitHist h;
    const int64_t m = c->m;
    sort_status_clear(u, (uint64_t)m);
    if (blockIdx.x * (int64_t)kT >= m) return;  // workgroup-uniform
    const uint64_t mask = (1ull << b) - 1;
    hist_clear(h, u.passes);
    for (int64_t e = blockIdx.x * (int64_t)kT + threadIdx.x; e < m; e += (int64_t)gridDim.x * kT) {
        const uint64_t k = keys[e];
        const uint32_t r = rank[k >> b], q = rank[k & mask];
        const uint64_t x = ((uint64_t)max(r, q) << b) | (uint64_t)min(r, q);
        keys[e] = x;
        hist_add(h, u.passes, x);
    }
    hist_flush(h, u);
}

#define BTC_LAUNCH(kernel, n, s, ...)                                                   \
    do {                                                                                \
        hipLaunchKernelGGL(kernel, dim3(grid_for(n)), dim3(kT), 0, s, __VA_ARGS__);     \
        BTC_CHECK_LAUNCH(#kernel);                                                      \
    } while (0)

// Kernels that end in same-address atomics (one per workgroup) run on at
// most kRedBlocks workgroups.
#define BTC_LAUNCH_RED(kernel, n, s, ...)                                                   \
    do {                                                                                \
        hipLaunchKernelGGL(kernel, dim3(std::min(grid_for(n), kRedBlocks)), dim3(kT), 0, s, __VA_ARGS__);     \
        BTC_CHECK_LAUNCH(#kernel);                                                      \
    } while (0)

}  // namespace

void canonicalise_device(const int32_t* src, const int32_t* dst, int64_t nnz, int32_t n, uint32_t flags,
                         hipStream_t s, btc_graph_s* g, const std::vector<int64_t>* segs,
                         std::vector<int64_t>* csegs) {
    BTC_REQUIRE(nnz < (int64_t)0xFFFFFFFFLL, BTC_ERR_OVERFLOW, "nnz %lld exceeds 2^32 - 1 pairs", (long long)nnz);
    const int nseg = segs ? (int)segs->size() - 1 : 0;
    if (segs) {
        BTC_REQUIRE(nseg >= 1 && csegs && (*segs)[0] == 0 && segs->back() == n, BTC_ERR_ARG,
                    "bad segments (%d segments over %d vertices)", nseg, n);
        for (int k = 0; k < nseg; ++k) BTC_REQUIRE((*segs)[k] <= (*segs)[k + 1], BTC_ERR_ARG, "segments not ascending");
    }
    // id range (and n when not given)
    int32_t h_lohi[2] = {INT_MAX, -1};
    {
        TmpBuf<int32_t> lohi;
        lohi.alloc(2, s);
        BTC_HIP(hipMemcpyAsync(lohi.p, h_lohi, 8, hipMemcpyHostToDevice, s));
        if (nnz) BTC_LAUNCH_RED(id_range_kernel, nnz, s, src, dst, nnz, lohi.p);
        BTC_HIP(hipMemcpyAsync(h_lohi, lohi.p, 8, hipMemcpyDeviceToHost, s));
        BTC_HIP(hipStreamSynchronize(s));
    }
    if (nnz == 0) h_lohi[0] = 0;
    BTC_REQUIRE(h_lohi[0] >= 0, BTC_ERR_ARG, "negative vertex id %d", h_lohi[0]);
    if (n <= 0) n = h_lohi[1] + 1;
    BTC_REQUIRE(h_lohi[1] < n, BTC_ERR_ARG, "vertex id %d >= n = %d", h_lohi[1], n);
    g->n_input = n;
    g->flags = flags;
    const int b = id_bits(n);
    const uint64_t sentinel = (1ull << (2 * b)) - 1;

    // oriented keys, sorted, deduplicated
    TmpBuf<uint64_t> ka, kb;
    ka.alloc((size_t)nnz, s);
    kb.alloc((size_t)nnz, s);
    if (nnz) BTC_LAUNCH(orient_kernel, nnz, s, src, dst, nnz, b, sentinel, ka.p);
    uint64_t* sorted = sort_u64(ka.p, kb.p, (size_t)nnz, 2 * b, s);
    uint64_t* other = sorted == ka.p ? kb.p : ka.p;
    int64_t m = 0;
    {
        TmpBuf<uint32_t> flag, pos;
        flag.alloc((size_t)nnz, s);
        pos.alloc((size_t)nnz + 1, s);
        if (nnz) BTC_LAUNCH(first_flag_kernel, nnz, s, sorted, nnz, sentinel, flag.p);
        exclusive_scan_u32(flag.p, pos.p, (size_t)nnz, s);
        uint32_t hm = 0;
        BTC_HIP(hipMemcpyAsync(&hm, pos.p + nnz, 4, hipMemcpyDeviceToHost, s));
        if (nnz) BTC_LAUNCH(compact_kernel, nnz, s, sorted, flag.p, pos.p, nnz, other);
        BTC_HIP(hipStreamSynchronize(s));
        m = hm;
    }
    uint64_t* keys = other;      // m unique oriented pairs, ascending
    uint64_t* spare = sorted;

    // order-preserving compaction of the used ids (none when no edge)
    int32_t nc = n;
    TmpBuf<uint32_t> newid;
    DevBuf<int32_t> labels;
    if ((flags & BTC_CANON_COMPACT) && m > 0) {
        TmpBuf<uint32_t> used;
        used.alloc((size_t)n, s);
        newid.alloc((size_t)n + 1, s);
        BTC_HIP(hipMemsetAsync(used.p, 0, (size_t)n * 4, s));
        BTC_LAUNCH(mark_used_kernel, m, s, keys, m, b, used.p);
        exclusive_scan_u32(used.p, newid.p, (size_t)n, s);
        uint32_t hn = 0;
        BTC_HIP(hipMemcpyAsync(&hn, newid.p + n, 4, hipMemcpyDeviceToHost, s));
        BTC_HIP(hipStreamSynchronize(s));
        nc = (int32_t)hn;
        labels.alloc_on((size_t)nc, s);
        BTC_LAUNCH(labels_kernel, n, s, used.p, newid.p, n, labels.p);
    } else {
        labels.alloc_on((size_t)n, s);
        BTC_LAUNCH(iota_kernel, n, s, labels.p, (int64_t)n);
    }
    const int bn = id_bits(nc);
    if (m) BTC_LAUNCH(relabel_kernel, m, s, keys, m, b, newid.p, bn);  // monotone: order kept
    // segment starts after compaction (the relabel is monotone, so every
    // segment stays one contiguous range)
    TmpBuf<uint32_t> dseg;
    if (segs) {
        std::vector<uint32_t> at(segs->begin(), segs->end()), cs(at.size());
        dseg.alloc(at.size(), s);
        BTC_HIP(hipMemcpyAsync(dseg.p, at.data(), at.size() * 4, hipMemcpyHostToDevice, s));
        if (newid.p) {
            TmpBuf<uint32_t> tmp;
            tmp.alloc(at.size(), s);
            hipLaunchKernelGGL(gather_kernel, dim3((unsigned)((at.size() + kT - 1) / kT)), dim3(kT), 0, s, newid.p,
                               dseg.p, (int)at.size(), tmp.p);
            BTC_CHECK_LAUNCH("gather_kernel");
            BTC_HIP(hipMemcpyAsync(dseg.p, tmp.p, at.size() * 4, hipMemcpyDeviceToDevice, s));
        }
        BTC_HIP(hipMemcpyAsync(cs.data(), dseg.p, cs.size() * 4, hipMemcpyDeviceToHost, s));
        BTC_HIP(hipStreamSynchronize(s));
        csegs->assign(cs.begin(), cs.end());
    }

    if (flags & BTC_CANON_DEGREE_ORDER) {
        TmpBuf<uint32_t> deg, k0, v0, k1, v1, rank;
        DevBuf<int32_t> lab2;
        uint32_t copies = m >= (int64_t)nc || nc <= kDegCopyIds ? kDegCopies : 1;
        k0.alloc((size_t)nc, s);
        v0.alloc((size_t)nc, s);
        if (!deg.try_alloc((size_t)nc * copies, s)) deg.alloc((size_t)nc * (copies = 1), s);
        BTC_HIP(hipMemsetAsync(deg.p, 0, (size_t)nc * copies * 4, s));
        if (m) {
            hipLaunchKernelGGL(degree_kernel, dim3(std::min(grid_for(m), kRedBlocks)), dim3(kT), 0, s, keys, m, bn, deg.p,
                               (size_t)nc, copies);
            BTC_CHECK_LAUNCH("degree_kernel");
        }
        BTC_LAUNCH(rank_keys_kernel, nc, s, deg.p, (size_t)nc, copies, nc, (uint32_t)nc, k0.p, v0.p);  // degrees are below nc
        deg.release();
        k1.alloc((size_t)nc, s);
        v1.alloc((size_t)nc, s);
        rank.alloc((size_t)nc, s);
        lab2.alloc_on((size_t)nc, s);
        bool alt = sort_pairs_u32(k0.p, v0.p, k1.p, v1.p, (size_t)nc, id_bits((int64_t)nc + 1), s);
        if (segs) {
            // then a stable sort by segment: (segment, -degree, id)
            uint32_t* ord = alt ? v1.p : v0.p;
            uint32_t* kk = alt ? k0.p : k1.p;  // free key buffer
            uint32_t* vv = alt ? v0.p : v1.p;  // free value buffer
            BTC_LAUNCH(segment_keys_kernel, nc, s, ord, nc, dseg.p, nseg, kk, vv);
            int sb = 1;
            while (sb < 32 && (1ll << sb) < (int64_t)nseg) ++sb;
            // sort (kk, vv) using (other key buffer, ord) as the spare pair
            uint32_t* kk2 = alt ? k1.p : k0.p;
            const bool alt2 = sort_pairs_u32(kk, vv, kk2, ord, (size_t)nc, sb, s);
            alt = alt2 ? (ord == v1.p) : (vv == v1.p);
        }
        BTC_LAUNCH(rank_scatter_kernel, nc, s, alt ? v1.p : v0.p, nc, rank.p, labels.p, lab2.p);
        if (m) BTC_LAUNCH(relabel_kernel, m, s, keys, m, bn, rank.p, bn);
        keys = sort_u64(keys, spare, (size_t)m, 2 * bn, s);
        labels.release_on(s);
        labels = std::move(lab2);
    }

    // CSR of L
    g->n = nc;
    g->m = m;
    g->d_rowptr.alloc_on((size_t)nc + 1, s);
    g->d_col.alloc_on((size_t)m + kColPad, s);
    BTC_LAUNCH(csr_kernel, std::max<int64_t>((int64_t)nc + 1, m + (int64_t)kColPad), s, keys, m, bn, nc,
               g->d_rowptr.p, g->d_col.p, (uint16_t*)nullptr, (uint32_t*)nullptr);
    g->d_labels = std::move(labels);

    // derived statistics (graph_finalize on the device)
    TmpBuf<unsigned long long> st;
    st.alloc(3, s);
    BTC_HIP(hipMemsetAsync(st.p, 0, 24, s));
    if (nc) BTC_LAUNCH_RED(stats_kernel, std::max<int64_t>(nc, m), s, g->d_rowptr.p, g->d_col.p, nc, m, st.p);
    unsigned long long h[3] = {0, 0, 0};
    BTC_HIP(hipMemcpyAsync(h, st.p, 24, hipMemcpyDeviceToHost, s));
    stream_wait(s);
    g->max_row = (int32_t)h[0];
    g->wedges = (int64_t)h[1];
    g->merge_work = (int64_t)h[2];
    g->on_host = false;
}

namespace {

// Grid of a capacity-sized launch: its workgroups stride over the live
// count, so a few per CU suffice.
unsigned cap_grid(int64_t cap) {
    return (unsigned)std::max<int64_t>(1, std::min<int64_t>((cap + kT - 1) / kT, 2048));
}

}  // namespace

#define CAP_LAUNCH(kernel, cap, s, ...)                                                \
    do {                                                                               \
        hipLaunchKernelGGL(kernel, dim3(cap_grid(cap)), dim3(kT), 0, s, __VA_ARGS__);  \
        BTC_CHECK_LAUNCH(#kernel);                                                     \
    } while (0)

// Kernels that end in atomics on a few addresses (reductions, digit totals).
#define CAP_LAUNCH_RED(kernel, cap, s, ...)                                                \
    do {                                                                                   \
        hipLaunchKernelGGL(kernel, dim3(std::min(cap_grid(cap), 2 * kCapRedBlocks)), dim3(kT), 0, s, __VA_ARGS__);  \
        BTC_CHECK_LAUNCH(#kernel);                                                         \
    } while (0)

int32_t* canonicalise_capacity(const CanonCap& c, hipStream_t s) {
    PipeCtl* ctl = c.ctl;
    const int64_t E = c.nnz_cap, N = c.n_cap;
    const int b = id_bits(N);
    const uint64_t sentinel = (1ull << (2 * b)) - 1;
    const Cnt m = Cnt::dev(&ctl->m), nc = Cnt::dev(&ctl->nc);
    const bool compact = (c.flags & BTC_CANON_COMPACT) != 0, groups = c.max_graphs > 1;
    const uint64_t seq_words = dseq_clear_words(c.seq->cap);
    hipLaunchKernelGGL(pipe_begin_kernel, dim3(std::min(cap_grid((int64_t)seq_words), kCapRedBlocks)), dim3(kT), 0, s,
                       ctl, static_cast<uint32_t*>(c.seq->p), seq_words, c.work, groups ? c.per_graph : nullptr,
                       (uint32_t)c.max_graphs);
    BTC_CHECK_LAUNCH("pipe_begin_kernel");

    // oriented keys, sorted, deduplicated
    const SortUse su = dseq_sort(*c.seq, 2 * b);
    CAP_LAUNCH_RED(orient_checked_kernel, E / 4 + 1, s, c.src, c.dst, ctl, c.n_cap, b, sentinel, c.ka, su);
    uint64_t* sorted = dsort_u64(c.ka, c.kb, (size_t)E, &ctl->nnz, su, s);
    uint64_t* keys = sorted == c.ka ? c.kb : c.ka;
    uint64_t* spare = sorted;
    with_tile_per(E, [&](auto per) {
        constexpr int PER = decltype(per)::value;
        CAP_LAUNCH(unique_kernel<PER>, E / PER + 1, s, sorted, ctl, c.n_cap, b, sentinel, keys,
                   compact ? c.used : nullptr, dseq_scan(*c.seq));
    });

    // order-preserving compaction of the used ids (ids keep b bits); the
    // graphs' ranges follow it; degrees
    int32_t* labels = c.lab0;
    if (compact)
        with_tile_per(N, [&](auto per) {
            constexpr int PER = decltype(per)::value;
            CAP_LAUNCH(newid_kernel<PER>, N / PER + 1, s, c.used, ctl, c.newid, labels, dseq_scan(*c.seq));
        });
    const bool by_degree = (c.flags & BTC_CANON_DEGREE_ORDER) != 0;
    hipLaunchKernelGGL(pipe_rekey_kernel, dim3(std::min(cap_grid(std::max(N, E)), 4 * kCapRedBlocks)), dim3(kT), 0, s,
                       keys, ctl, b, compact ? c.newid : nullptr, labels, c.segs, groups ? c.csegs : nullptr,
                       by_degree ? c.deg : nullptr, (size_t)N);
    BTC_CHECK_LAUNCH("pipe_rekey_kernel");

    if (by_degree) {
        // keys N - 1 - degree < 2^b: descending degree, ties by id
        int kb = b;  // key bits: degree rank, then (several graphs) the graph
        if (groups) {
            int gb = 1;
            while ((1 << gb) < c.max_graphs) ++gb;
            BTC_REQUIRE(b + gb <= 32, BTC_ERR_OVERFLOW, "%d ids and %d graphs exceed 32-bit relabel keys", c.n_cap,
                        c.max_graphs);
            kb = b + gb;
        }
        const SortUse ru = dseq_sort(*c.seq, kb);
        CAP_LAUNCH_RED(pipe_rank_keys_kernel, N, s, c.deg, (size_t)N, ctl, groups ? c.csegs : nullptr,
                       (uint32_t)(N - 1), b, c.k0, c.v0, ru);
        const bool alt = dsort_pairs_u32(c.k0, c.v0, c.k1, c.v1, (size_t)N, &ctl->nc, ru, s);
        CAP_LAUNCH(rank_scatter_kernel, N, s, alt ? c.v1 : c.v0, nc, c.rank, labels, c.lab1);
        const SortUse ku = dseq_sort(*c.seq, 2 * b);
        CAP_LAUNCH_RED(pipe_relabel_kernel, E, s, keys, ctl, b, c.rank, ku);
        keys = dsort_u64(keys, spare, (size_t)E, &ctl->m, ku, s);
        labels = c.lab1;
    }

    // CSR of L (with its 16-bit copy and every entry's row) and its statistics
    CAP_LAUNCH(csr_kernel, std::max(N + 1, E + (int64_t)kColPad), s, keys, m, b, nc, c.rowptr, c.col, c.col16, c.erow);
    hipLaunchKernelGGL(stats_kernel, dim3(std::min(cap_grid(std::max(N, E)), kCapRedBlocks)), dim3(kT), 0, s, c.rowptr,
                       c.col, nc, m, ctl->rs);
    BTC_CHECK_LAUNCH("stats_kernel");
    return labels;
}

void ensure_host(btc_graph_s* g) {
    if (g->on_host) return;
    std::vector<uint32_t> rp((size_t)g->n + 1);
    std::vector<int32_t> col((size_t)g->m), labels((size_t)g->n);
    BTC_HIP(hipMemcpy(rp.data(), g->d_rowptr.p, rp.size() * 4, hipMemcpyDeviceToHost));
    if (g->m) BTC_HIP(hipMemcpy(col.data(), g->d_col.p, (size_t)g->m * 4, hipMemcpyDeviceToHost));
    if (g->n) BTC_HIP(hipMemcpy(labels.data(), g->d_labels.p, (size_t)g->n * 4, hipMemcpyDeviceToHost));
    g->rowptr.assign(rp.begin(), rp.end());
    g->col.swap(col);
    g->labels.swap(labels);
    g->on_host = true;
}

}  // namespace btcx

extern "C" {

int btc_graph_from_coo_device(const int32_t* src, const int32_t* dst, int64_t nnz, int32_t n, uint32_t flags,
                              void* stream, btc_graph* out) {
    return btcx::guard([&] {
        BTC_REQUIRE(out, BTC_ERR_ARG, "out is NULL");
        *out = nullptr;
        BTC_REQUIRE(nnz >= 0, BTC_ERR_ARG, "nnz %lld < 0", (long long)nnz);
        BTC_REQUIRE(nnz == 0 || (src && dst), BTC_ERR_ARG, "src/dst is NULL");
        BTC_REQUIRE((flags & ~BTC_CANON_DEFAULT) == 0, BTC_ERR_ARG, "unknown flags 0x%x", flags);
        auto g = std::make_unique<btc_graph_s>();
        btcx::canonicalise_device(src, dst, nnz, n, flags, btcx::as_stream(stream), g.get(), nullptr, nullptr);
        *out = g.release();
    });
}

}  // extern "C"
