// Device planner: the wedge-kernel plan of a graph whose L is resident in
// HBM, built by kernels, radix sorts and scans instead of host loops.
//
// The plan has the same contents as the host planner's (engine.hip,
// classify_dense + build_wedge_lists): dense mask tiles (popcount > tau)
// listed for the tile kernel; for every other edge (i, j) of L the prefix
// of row i in front of j clipped to [min N_L(j), max N_L(j)], with its
// hub-core bitmap choice; lists grouped by pivot j; work items of about
// `chunk` checks, workgroup items then wave items, each class by work.  Two
// details differ and neither changes a count: lists of one pivot are in
// edge order (a stable radix sort by pivot), and a pivot's lists are cut
// where the running cost crosses a multiple of `chunk` rather than
// greedily.
#include "devtile.h"
#include "internal.h"

namespace btcx {
namespace {

constexpr int kT = 256;
constexpr unsigned kRedBlocks = 1024;    // eager reductions
constexpr unsigned kCapRedBlocks = 256;  // capacity-sized reductions: about one per CU

unsigned grid_for(int64_t n) {
    const int64_t g = (n + kT - 1) / kT;
    return (unsigned)std::max<int64_t>(1, std::min<int64_t>(g, 65536));
}

int id_bits(int64_t n) {
    int b = 1;
    while (b < 32 && (1ll << b) < n) ++b;
    return b;
}

#define GS_LOOP(i, n) for (int64_t i = blockIdx.x * (int64_t)kT + threadIdx.x; i < (n); i += (int64_t)gridDim.x * kT)

#define BTC_LAUNCH(kernel, n, s, ...)                                               \
    do {                                                                            \
        hipLaunchKernelGGL(kernel, dim3(grid_for(n)), dim3(kT), 0, s, __VA_ARGS__); \
        BTC_CHECK_LAUNCH(#kernel);                                                  \
    } while (0)

// Kernels that end in same-address atomics (one per workgroup) run on at
// most kRedBlocks workgroups.
#define BTC_LAUNCH_RED(kernel, n, s, ...)                                               \
    do {                                                                            \
        hipLaunchKernelGGL(kernel, dim3(std::min(grid_for(n), kRedBlocks)), dim3(kT), 0, s, __VA_ARGS__); \
        BTC_CHECK_LAUNCH(#kernel);                                                  \
    } while (0)

// The passes over entries and lists: bound by the latency of their dependent
// loads, so they fill the chip twice over.
#define BTC_LAUNCH_CLIP(kernel, n, s, ...)                                                  \
    do {                                                                                    \
        hipLaunchKernelGGL(kernel, dim3(std::min(grid_for(n), 4 * kRedBlocks)), dim3(kT), 0, s, __VA_ARGS__); \
        BTC_CHECK_LAUNCH(#kernel);                                                          \
    } while (0)

// First index in [lo, hi) of a[] with a[x] >= v (a ascending).
template <class T>
__device__ __forceinline__ uint32_t lower_bound_dev(const T* a, uint32_t lo, uint32_t hi, T v) {
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (a[mid] < v) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

template <class T>
__device__ __forceinline__ uint32_t upper_bound_dev(const T* a, uint32_t lo, uint32_t hi, T v) {
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (a[mid] <= v) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// erow[e] = row of entry e: one wave per row, lanes stride over its entries.
__global__ void edge_rows_kernel(const uint32_t* __restrict__ rowptr, Cnt n_, uint32_t* __restrict__ erow) {
    const int64_t n = (int64_t)n_.get();
    const int64_t waves = ((int64_t)gridDim.x * kT) >> 6;
    const int lane = threadIdx.x & 63;
    for (int64_t i = (blockIdx.x * (int64_t)kT + threadIdx.x) >> 6; i < n; i += waves)
        for (uint32_t p = rowptr[i] + lane; p < rowptr[i + 1]; p += 64) erow[p] = (uint32_t)i;
}

// Dense mask tiles: flag[t] = popcount > tau; dense edges summed.
__global__ void dense_tiles_kernel(const uint32_t* __restrict__ pop, uint32_t nblk, int tau,
                                   uint32_t* __restrict__ flag, unsigned long long* __restrict__ dense_edges) {
    uint64_t sum = 0;
    GS_LOOP(t, nblk) {
        const bool d = (int)pop[t] > tau;
        flag[t] = d;
        sum += d ? pop[t] : 0u;
    }
    __shared__ uint64_t lds[kT / 64];
    sum = block_sum_u64<kT>(sum, lds);
    if (threadIdx.x == 0 && sum) atomicAdd(dense_edges, (unsigned long long)sum);
}

__global__ void select_kernel(const uint32_t* __restrict__ flag, const uint32_t* __restrict__ pos, Cnt n_,
                              uint32_t* __restrict__ out) {
    const int64_t n = (int64_t)n_.get();
    GS_LOOP(t, n) if (flag[t]) out[pos[t]] = (uint32_t)t;
}

// dense[e] = the edge lies in a dense mask tile of the Bit-BSR.
__global__ void dense_edges_kernel(const int32_t* __restrict__ col, const uint32_t* __restrict__ erow, int64_t m,
                                   int K, const uint32_t* __restrict__ indptr, const uint32_t* __restrict__ indices,
                                   const uint32_t* __restrict__ pop, int tau, uint8_t* __restrict__ dense) {
    GS_LOOP(e, m) {
        const uint32_t I = erow[e] / 16, jc = (uint32_t)col[e] / (uint32_t)K;
        const uint32_t t0 = indptr[I], t1 = indptr[I + 1];  // no tiles: no dense tile in the row block
        dense[e] = t0 != t1 && (int)pop[lower_bound_dev(indices, t0, t1, jc)] > tau;
    }
}

// Clipped prefix of entry q (row i, pivot j = col[q]) as in the host
// planner; false when nothing in it can match.
__device__ __forceinline__ bool clip(const uint32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                                     uint32_t i, uint32_t q, uint32_t& s0, uint32_t& s1) {
    const uint32_t j = (uint32_t)col[q];
    const uint32_t r0 = rowptr[i], t0 = rowptr[j], t1 = rowptr[j + 1];
    if (t1 == t0 || q == r0) return false;
    const int32_t lo = col[t0], hi = col[t1 - 1];
    s0 = lower_bound_dev(col, r0, q, lo);
    s1 = upper_bound_dev(col, s0, q, hi);
    return s1 > s0;
}

// The list of entry q (row i, whose ids below C end at ce and whose core
// bitmap is rb): its record {s0, s_noncore, s1, bitmap}; false when it is
// empty.
__device__ __forceinline__ bool list_record(const uint32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                                            uint32_t i, uint32_t q, uint32_t ce, uint32_t rb, uint32_t C, uint4& r) {
    uint32_t s0, s1;
    if (!clip(rowptr, col, i, q, s0, s1)) return false;
    r = make_uint4(s0, s0, s1, kNoBitmap);
    if (rb != kNoBitmap) {
        const uint32_t j = (uint32_t)col[q];
        const uint32_t lo = (uint32_t)col[rowptr[j]], hi = (uint32_t)col[rowptr[j + 1] - 1];
        if ((lo & ~127u) < C) {
            const uint32_t c1 = min(s1, ce), ids = c1 > s0 ? c1 - s0 : 0u, w = core_words(lo, hi, C);
            if (take_core_bitmap(ids, w)) {
                r.y = max(s0, ce);
                r.w = rb;
            }
        }
    }
    return true;
}

// Pass over the entries of L: list flag and record of every entry (rec[q]
// where flagged), sparse edge count and merge work.  Records are made here,
// where neighbouring entries share a row's cache lines, and fetched once
// after the sort by pivot: made in list order, each list searched a random
// row twice (R-MAT 2^20, 12 M lists: 1666 us there; here 72 us more than the
// flags alone, and 525 us to fetch them).
__global__ void clip_kernel(const uint32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                            const uint32_t* __restrict__ erow, const uint8_t* __restrict__ dense, int64_t m,
                            const uint32_t* __restrict__ cend, const uint32_t* __restrict__ has,
                            const uint32_t* __restrict__ rbi, uint32_t C, uint32_t* __restrict__ flag,
                            uint4* __restrict__ rec, unsigned long long* __restrict__ stats) {
    uint64_t se = 0, sw = 0;
    GS_LOOP(q, m) {
        uint32_t f = 0;
        if (!dense || !dense[q]) {
            const uint32_t i = erow[q], j = (uint32_t)col[q];
            ++se;
            sw += (rowptr[i + 1] - rowptr[i]) + (rowptr[j + 1] - rowptr[j]);
            uint4 r;
            f = list_record(rowptr, col, i, (uint32_t)q, cend[i], has[i] ? rbi[i] : kNoBitmap, C, r);
            if (f) rec[q] = r;
        }
        flag[q] = f;
    }
    __shared__ uint64_t lds[kT / 64];
    se = block_sum_u64<kT>(se, lds);
    sw = block_sum_u64<kT>(sw, lds);
    if (threadIdx.x == 0) {
        if (se) atomicAdd(&stats[0], (unsigned long long)se);
        if (sw) atomicAdd(&stats[1], (unsigned long long)sw);
    }
}

__global__ void list_keys_kernel(const uint32_t* __restrict__ flag, const uint32_t* __restrict__ pos,
                                 const int32_t* __restrict__ col, Cnt m_, uint32_t* __restrict__ key,
                                 uint32_t* __restrict__ val) {
    const int64_t m = (int64_t)m_.get();
    GS_LOOP(q, m) if (flag[q]) {
        key[pos[q]] = (uint32_t)col[q];
        val[pos[q]] = (uint32_t)q;
    }
}

// off[j] = first list of pivot j (j = 0..n) in the pivot-sorted keys.
__global__ void pivot_offsets_kernel(const uint32_t* __restrict__ key, Cnt ne_, Cnt n_,
                                     uint32_t* __restrict__ off) {
    const uint32_t ne = (uint32_t)ne_.get();
    const int64_t n = (int64_t)n_.get();
    GS_LOOP(j, (int64_t)n + 1) off[j] = lower_bound_dev(key, 0u, ne, (uint32_t)j);
}

// Core ids (< C) per row; rows with at least kCoreRowMin get a bitmap.
__global__ void core_rows_kernel(const uint32_t* __restrict__ rowptr, const int32_t* __restrict__ col, Cnt n_,
                                 uint32_t C, uint32_t* __restrict__ cend, uint32_t* __restrict__ has) {
    const int64_t n = (int64_t)n_.get();
    GS_LOOP(i, n) {
        const uint32_t r0 = rowptr[i];
        const uint32_t c = lower_bound_dev(col, r0, rowptr[i + 1], (int32_t)C);
        cend[i] = c;
        has[i] = c - r0 >= kCoreRowMin;
    }
}

// Core bitmaps, a wave per row that has one: lane w % 64 owns word w, taken
// 64 words (2048 ids) at a time from the row's ids below C, so a bitmap is
// cleared, set and written in one pass without atomics.
// (R-MAT 2^20: 95 us; with a memset and an atomic per id 164 us and the memset).
// has (NULL: rbi says it, kNoBitmap) = the row has a bitmap.
__global__ __launch_bounds__(kT) void core_fill_kernel(const uint32_t* __restrict__ rowptr,
                                                       const int32_t* __restrict__ col,
                                                       const uint32_t* __restrict__ cend,
                                                       const uint32_t* __restrict__ has,
                                                       const uint32_t* __restrict__ rbi, Cnt n_, uint32_t C,
                                                       uint32_t* __restrict__ rowbits) {
    const int64_t n = n_.get(), waves = ((int64_t)gridDim.x * kT) >> 6;
    const uint32_t lane = threadIdx.x & 63, CW = C / 32;
    for (int64_t i = (blockIdx.x * (int64_t)kT + threadIdx.x) >> 6; i < n; i += waves) {
        if (has ? !has[i] : rbi[i] == kNoBitmap) continue;
        uint32_t* b = rowbits + (size_t)rbi[i] * CW;
        const uint32_t p1 = cend[i];
        uint32_t p = rowptr[i];
        for (uint32_t w0 = 0; w0 < CW; w0 += 64) {
            uint32_t word = 0;
            // ids of this span, 64 at a time, each lane picking its word's
            while (p < p1) {
                const uint32_t at = p + lane;
                const uint32_t id = at < p1 ? (uint32_t)col[at] : 0xFFFFFFFFu;
                const uint64_t in = __ballot(id < (w0 + 64) * 32);
                const int cnt = __popcll(in);
                for (int k = 0; k < cnt; ++k) {
                    const uint32_t kid = (uint32_t)__builtin_amdgcn_readlane((int)id, k);
                    word |= (kid >> 5) - w0 == lane ? 1u << (kid & 31u) : 0u;
                }
                p += (uint32_t)cnt;
                if (cnt < 64) break;
            }
            if (w0 + lane < CW) b[w0 + lane] = word;
        }
    }
}

// Record of every pivot-sorted list e (see the wedge kernel's scan_lists), its
// row, and its cost (ids looked up + core words ANDed).
__global__ void records_kernel(const uint32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                               const uint32_t* __restrict__ erow, const uint32_t* __restrict__ key,
                               const uint32_t* __restrict__ val, int64_t ne, const uint4* __restrict__ rec, uint32_t C,
                               uint4* __restrict__ lst, int32_t* __restrict__ ur, uint64_t* __restrict__ cost,
                               unsigned long long* __restrict__ ncore, unsigned long long* __restrict__ nnarrow) {
    uint64_t nc = 0, nn = 0;
    GS_LOOP(e, ne) {
        const uint32_t q = val[e], j = key[e];
        const uint4 r = rec[q];
        const uint32_t lo = (uint32_t)col[rowptr[j]], hi = (uint32_t)col[rowptr[j + 1] - 1];
        const uint32_t ids = r.z > r.y ? r.z - r.y : 0u;
        lst[e] = r;
        ur[e] = (int32_t)erow[q];
        cost[e] = (uint64_t)ids + (r.w != kNoBitmap ? core_words(lo, hi, C) : 0u);
        nc += r.w != kNoBitmap;
        nn += hi < kNarrowIds ? ids : 0u;
    }
    __shared__ uint64_t lds[kT / 64];
    nc = block_sum_u64<kT>(nc, lds);
    nn = block_sum_u64<kT>(nn, lds);
    if (threadIdx.x == 0 && nc) atomicAdd(ncore, (unsigned long long)nc);
    if (threadIdx.x == 0 && nn) atomicAdd(nnarrow, (unsigned long long)nn);
}

__device__ __forceinline__ bool pivot_small(const uint32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                                            const uint32_t* __restrict__ off, uint32_t j) {
    const uint32_t t0 = rowptr[j], t1 = rowptr[j + 1];
    return wave_pivot(off[j + 1] - off[j], (uint32_t)col[t0], (uint32_t)col[t1 - 1], t1 - t0);
}

// start[e] = list e opens a work item: the pivot's first list, or (large
// pivots) the running cost crosses a multiple of chunk.
__global__ void item_start_kernel(const uint32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                                  const uint32_t* __restrict__ key, const uint32_t* __restrict__ off,
                                  const uint64_t* __restrict__ P, int64_t ne, uint64_t chunk,
                                  uint32_t* __restrict__ start) {
    GS_LOOP(e, ne) {
        const uint32_t j = key[e], eb = off[j];
        uint32_t st = e == eb;
        if (!st && !pivot_small(rowptr, col, off, j)) st = (P[e] - P[eb]) / chunk != (P[e - 1] - P[eb]) / chunk;
        start[e] = st;
    }
}

// Item k = lists [first[k], first[k + 1]); sort key puts workgroup items
// before wave items before tiny items, each by descending work.
__global__ void items_kernel(const uint32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                             const uint32_t* __restrict__ key, const uint32_t* __restrict__ off,
                             const uint64_t* __restrict__ P, const uint32_t* __restrict__ first, Cnt nitems_,
                             Cnt ne_, bool use_tiny, bool tiny_all, uint4* __restrict__ tmp_items,
                             uint32_t* __restrict__ skey, uint32_t* __restrict__ sval,
                             unsigned long long* __restrict__ stats) {
    const uint32_t nitems = (uint32_t)nitems_.get();
    const uint32_t ne = (uint32_t)ne_.get();
    uint64_t words = 0, small_items = 0, tiny_items = 0;
    GS_LOOP(k, nitems) {
        const uint32_t eb = first[k], ee = k + 1 < nitems ? first[k + 1] : ne;
        const uint32_t j = key[eb];
        const uint32_t t0 = rowptr[j], t1 = rowptr[j + 1];
        const uint64_t w = P[ee] - P[eb];
        const uint32_t w32 = (uint32_t)min(w, (uint64_t)0xFFFFFFFFu);
        const uint32_t lo = (uint32_t)col[t0], hi = (uint32_t)col[t1 - 1];
        const bool small = pivot_small(rowptr, col, off, j);
        const bool tiny = use_tiny && small && tiny_pivot(off[j + 1] - off[j], lo, hi, t1 - t0, tiny_all);
        tmp_items[2 * k] = make_uint4(t0, t1, eb, ee);
        tmp_items[2 * k + 1] = make_uint4(lo, hi, w32, 0u);
        const uint32_t cls = tiny ? 2u : small ? 1u : 0u;
        const uint32_t w30 = (uint32_t)min(w, (uint64_t)0x3FFFFFFFu);
        skey[k] = (cls << 30) | (0x3FFFFFFFu - w30);
        sval[k] = (uint32_t)k;
        words += t1 - t0;
        small_items += small;
        tiny_items += tiny;
    }
    __shared__ uint64_t lds[kT / 64];
    words = block_sum_u64<kT>(words, lds);
    small_items = block_sum_u64<kT>(small_items, lds);
    tiny_items = block_sum_u64<kT>(tiny_items, lds);
    if (threadIdx.x == 0) {
        if (words) atomicAdd(&stats[0], (unsigned long long)words);
        if (small_items) atomicAdd(&stats[1], (unsigned long long)small_items);
        if (tiny_items) atomicAdd(&stats[3], (unsigned long long)tiny_items);
    }
}

__global__ void place_items_kernel(const uint4* __restrict__ tmp_items, const uint32_t* __restrict__ order,
                                   int64_t nitems, uint4* __restrict__ items) {
    GS_LOOP(r, nitems) {
        const uint32_t k = order[r];
        items[2 * r] = tmp_items[2 * k];
        items[2 * r + 1] = tmp_items[2 * k + 1];
    }
}

// ------------------------------------------------- capturable form kernels
// Rows of L: the end of their ids below C (cend) and the index of their core
// bitmap (rbi; kNoBitmap for a row of fewer than kCoreRowMin of them; numbered
// in no particular order, one atomic a workgroup).
__global__ __launch_bounds__(kT) void pipe_rows_kernel(const uint32_t* __restrict__ rowptr,
                                                       const int32_t* __restrict__ col, PipeCtl* __restrict__ c,
                                                       uint32_t C, uint32_t* __restrict__ cend,
                                                       uint32_t* __restrict__ rbi) {
    __shared__ uint32_t s_has[kT / 64], s_base;
    const uint32_t lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int64_t n = c->nc;
    for (int64_t base = blockIdx.x * (int64_t)kT; base < n; base += (int64_t)gridDim.x * kT) {
        const int64_t r = base + threadIdx.x;
        bool has = false;
        if (r < n) {
            const uint32_t r0 = rowptr[r], ce = lower_bound_dev(col, r0, rowptr[r + 1], (int32_t)C);
            cend[r] = ce;
            has = ce - r0 >= kCoreRowMin;
        }
        const uint64_t some = __ballot(has);
        if (lane == 0) s_has[wid] = (uint32_t)__popcll(some);
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t t = 0;
            for (int k = 0; k < kT / 64; ++k) t += s_has[k];
            s_base = t ? atomicAdd(&c->nbm, t) : 0u;
        }
        __syncthreads();
        if (r < n) {
            uint32_t at = s_base + (uint32_t)__popcll(some & ((1ull << lane) - 1));
            for (uint32_t k = 0; k < wid; ++k) at += s_has[k];
            rbi[r] = has ? at : kNoBitmap;
        }
        __syncthreads();
    }
}

// Entries of L in tiles: those with a list (a non-empty clipped prefix) go
// to (pivot, entry) pairs in entry order, the list's record to rec[entry],
// where the entries of a row share its cache lines; the sort by pivot then
// moves 8 bytes a list and the records are fetched once, instead of every
// list's two searches of a random row (24 R-MAT graphs, 3.3 M entries: this
// kernel and the next 270 us against 490 us for flags, scan, pairs, records,
// costs and their scan as kernels of their own).  ne = lists.
template <int PER>
__global__ __launch_bounds__(kT) void pipe_clip_kernel(const uint32_t* __restrict__ rowptr,
                                                       const int32_t* __restrict__ col,
                                                       const uint32_t* __restrict__ erow,
                                                       const uint32_t* __restrict__ cend,
                                                       const uint32_t* __restrict__ rbi, uint32_t C,
                                                       PipeCtl* __restrict__ c, uint32_t* __restrict__ key,
                                                       uint32_t* __restrict__ val, uint4* __restrict__ rec, SortUse su,
                                                       ScanUse u) {
    __shared__ DigitHist h;
    __shared__ uint32_t lds[4 * PER + 2];
    __shared__ uint32_t s_tile;
    const uint32_t m = c->m;
    sort_status_clear(su, m);  // at most m lists
    constexpr uint32_t kTile = kT * PER;
    const uint32_t nt = (uint32_t)(((uint64_t)m + kTile - 1) / kTile);
    if (blockIdx.x >= nt) return;  // workgroup-uniform
    hist_clear(h, su.passes);
    for (TileLoop l(u.ticket, nt, &s_tile); l.next();) {
        uint32_t f[PER], pos[PER];
#pragma unroll
        for (int x = 0; x < PER; ++x) {
            const uint64_t q = (uint64_t)l.t * kTile + x * kT + threadIdx.x;
            f[x] = 0;
            if (q >= m) continue;
            const uint32_t i = erow[q];
            uint4 r;
            f[x] = list_record(rowptr, col, i, (uint32_t)q, cend[i], rbi[i], C, r);
            if (f[x]) rec[q] = r;
        }
        const uint64_t tot = tile_offsets<uint32_t, PER>(f, pos, lds, u, l.t);
        if (l.t == nt - 1 && threadIdx.x == 0) c->ne = (uint32_t)tot;
#pragma unroll
        for (int x = 0; x < PER; ++x) {
            if (!f[x]) continue;
            const uint32_t q = l.t * kTile + x * kT + threadIdx.x, j = (uint32_t)col[q];
            key[pos[x]] = j;
            val[pos[x]] = q;
            hist_add(h, su.passes, j);
        }
    }
    hist_flush(h, su);
}

// The lists by pivot: records, rows, the running cost P and the range of every
// pivot that has lists.
template <int PER>
__global__ __launch_bounds__(kT) void pipe_lists_kernel(const uint32_t* __restrict__ rowptr,
                                                        const int32_t* __restrict__ col,
                                                        const uint32_t* __restrict__ erow, uint32_t C,
                                                        PipeCtl* __restrict__ c, const uint32_t* __restrict__ key,
                                                        const uint32_t* __restrict__ val,
                                                        const uint4* __restrict__ rec, uint32_t* __restrict__ off,
                                                        uint32_t* __restrict__ oend, uint4* __restrict__ lst,
                                                        int32_t* __restrict__ ur, uint64_t* __restrict__ P,
                                                        ScanUse u) {
    __shared__ uint64_t lds[4 * PER + 2];
    __shared__ uint64_t red[kT / 64];
    __shared__ uint32_t s_tile;
    const uint32_t ne = c->ne;
    constexpr uint32_t kTile = kT * PER;
    const uint32_t nt = (uint32_t)(((uint64_t)ne + kTile - 1) / kTile);
    uint64_t nc = 0, nn = 0;
    for (TileLoop l(u.ticket, nt, &s_tile); l.next();) {
        uint64_t v[PER], at[PER];
#pragma unroll
        for (int x = 0; x < PER; ++x) {
            const uint64_t e = (uint64_t)l.t * kTile + x * kT + threadIdx.x;
            v[x] = 0;
            if (e >= ne) continue;
            const uint32_t j = key[e], q = val[e];
            const uint4 r = rec[q];
            const uint32_t lo = (uint32_t)col[rowptr[j]], hi = (uint32_t)col[rowptr[j + 1] - 1];
            const uint32_t ids = r.z > r.y ? r.z - r.y : 0u;
            lst[e] = r;
            ur[e] = (int32_t)erow[q];
            v[x] = (uint64_t)ids + (r.w != kNoBitmap ? core_words(lo, hi, C) : 0u);
            nc += r.w != kNoBitmap;
            nn += hi < kNarrowIds ? ids : 0u;
            if (e == 0 || key[e - 1] != j) off[j] = (uint32_t)e;
            if (e + 1 == ne || key[e + 1] != j) oend[j] = (uint32_t)e + 1;
        }
        const uint64_t tot = tile_offsets<uint64_t, PER>(v, at, lds, u, l.t);
        if (l.t == nt - 1 && threadIdx.x == 0) {
            P[ne] = tot;
            c->checks = tot;
        }
#pragma unroll
        for (int x = 0; x < PER; ++x) {
            const uint64_t e = (uint64_t)l.t * kTile + x * kT + threadIdx.x;
            if (e < ne) P[e] = at[x];
        }
    }
    __syncthreads();
    nc = block_sum_u64<kT>(nc, red);
    nn = block_sum_u64<kT>(nn, red);
    if (threadIdx.x == 0) {
        if (nc) atomicAdd(&c->st[3], (unsigned long long)nc);
        if (nn) atomicAdd(&c->st[6], (unsigned long long)nn);
    }
}

// List e opens a work item: the pivot's first list, or (pivots of more than
// a wave's worth) where the running cost crosses a multiple of the cut, about
// target_items items in all and at least 8192 checks each.  first[k] = the
// list that opens item k.
template <int PER>
__global__ __launch_bounds__(kT) void pipe_first_kernel(const uint32_t* __restrict__ rowptr,
                                                        const int32_t* __restrict__ col, PipeCtl* __restrict__ c,
                                                        const uint32_t* __restrict__ key,
                                                        const uint32_t* __restrict__ off,
                                                        const uint32_t* __restrict__ oend,
                                                        const uint64_t* __restrict__ P, uint64_t target_items,
                                                        uint32_t* __restrict__ first, ScanUse u) {
    __shared__ uint32_t lds[4 * PER + 2];
    __shared__ uint32_t s_tile;
    const uint32_t ne = c->ne;
    const uint64_t chunk = max((uint64_t)8192, ((uint64_t)c->checks + target_items - 1) / target_items);
    constexpr uint32_t kTile = kT * PER;
    const uint32_t nt = (uint32_t)(((uint64_t)ne + kTile - 1) / kTile);
    for (TileLoop l(u.ticket, nt, &s_tile); l.next();) {
        uint32_t f[PER], pos[PER];
#pragma unroll
        for (int x = 0; x < PER; ++x) {
            const uint64_t e = (uint64_t)l.t * kTile + x * kT + threadIdx.x;
            f[x] = 0;
            if (e >= ne) continue;
            const uint32_t j = key[e], eb = off[j];
            f[x] = e == eb;
            if (!f[x]) {
                const uint32_t t0 = rowptr[j], t1 = rowptr[j + 1];
                if (!wave_pivot(oend[j] - eb, (uint32_t)col[t0], (uint32_t)col[t1 - 1], t1 - t0))
                    f[x] = (P[e] - P[eb]) / chunk != (P[e - 1] - P[eb]) / chunk;
            }
        }
        const uint64_t tot = tile_offsets<uint32_t, PER>(f, pos, lds, u, l.t);
        if (l.t == nt - 1 && threadIdx.x == 0) c->nitems = (uint32_t)tot;
#pragma unroll
        for (int x = 0; x < PER; ++x)
            if (f[x]) first[pos[x]] = l.t * kTile + x * kT + threadIdx.x;
    }
}

// Bucket of an item's class and work: workgroup items before wave items, by
// half octaves of work, heaviest first.
__device__ __forceinline__ uint32_t item_bucket(bool small, uint64_t w) {
    const uint32_t len = w ? 64 - __clzll(w) : 0u;
    const uint32_t half = len >= 2 ? (uint32_t)(w >> (len - 2)) & 1u : 0u;
    return ((small ? 1u : 0u) << 6) | (63u - min(63u, 2 * len + half));
}

// Items per bucket; pivot row words and wave items (st[4], st[5]).
__global__ __launch_bounds__(kT) void pipe_item_keys_kernel(const uint32_t* __restrict__ rowptr,
                                                            const int32_t* __restrict__ col, PipeCtl* __restrict__ c,
                                                            const uint32_t* __restrict__ key,
                                                            const uint32_t* __restrict__ off,
                                                            const uint32_t* __restrict__ oend,
                                                            const uint64_t* __restrict__ P,
                                                            const uint32_t* __restrict__ first,
                                                            uint32_t* __restrict__ skey,
                                                            uint32_t* __restrict__ totals) {
    __shared__ uint32_t h[kDigits];
    __shared__ uint64_t red[kT / 64];
    const uint32_t nitems = c->nitems, ne = c->ne;
    if (blockIdx.x * kT >= nitems) return;  // workgroup-uniform
    h[threadIdx.x] = 0;
    __syncthreads();
    uint64_t words = 0, small_items = 0;
    GS_LOOP(k, nitems) {
        const uint32_t eb = first[k], ee = k + 1 < nitems ? first[k + 1] : ne, j = key[eb];
        const uint32_t t0 = rowptr[j], t1 = rowptr[j + 1];
        const bool small = wave_pivot(oend[j] - off[j], (uint32_t)col[t0], (uint32_t)col[t1 - 1], t1 - t0);
        const uint32_t s = item_bucket(small, P[ee] - P[eb]);
        skey[k] = s;
        atomicAdd(&h[s], 1u);
        words += t1 - t0;
        small_items += small;
    }
    __syncthreads();
    const uint32_t cnt = h[threadIdx.x];
    if (cnt) atomicAdd(&totals[threadIdx.x], cnt);
    words = block_sum_u64<kT>(words, red);
    small_items = block_sum_u64<kT>(small_items, red);
    if (threadIdx.x == 0) {
        if (words) atomicAdd(&c->st[4], (unsigned long long)words);
        if (small_items) atomicAdd(&c->st[5], (unsigned long long)small_items);
    }
}

// The items to their buckets (in no particular order within one), each with
// its graph when csegs is set (the last one whose rows start at or before its
// pivot row); workgroup 0 records the launch's item counts.
__global__ __launch_bounds__(kT) void pipe_place_kernel(const uint32_t* __restrict__ rowptr,
                                                        const int32_t* __restrict__ col, PipeCtl* __restrict__ c,
                                                        const uint32_t* __restrict__ key,
                                                        const uint64_t* __restrict__ P,
                                                        const uint32_t* __restrict__ first,
                                                        const uint32_t* __restrict__ skey,
                                                        const uint32_t* __restrict__ totals,
                                                        uint32_t* __restrict__ cursors,
                                                        const uint32_t* __restrict__ csegs,
                                                        uint4* __restrict__ items) {
    __shared__ uint32_t start[kDigits], h[kDigits], wsum[kT / 64];
    const uint32_t nitems = c->nitems, ne = c->ne, graphs = c->graphs;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        c->item_counts[0] = nitems - (uint32_t)c->st[5];
        c->item_counts[1] = nitems;
    }
    if (blockIdx.x * kT >= nitems) return;  // workgroup-uniform
    const uint32_t lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    uint32_t x = totals[threadIdx.x];
    const uint32_t own = x;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)x, o);
        if ((int)lane >= o) x += y;
    }
    if (lane == 63) wsum[wid] = x;
    __syncthreads();
    for (uint32_t k = 0; k < wid; ++k) x += wsum[k];
    start[threadIdx.x] = x - own;
    for (uint64_t k0 = (uint64_t)blockIdx.x * kT; k0 < nitems; k0 += (uint64_t)gridDim.x * kT) {
        h[threadIdx.x] = 0;
        __syncthreads();
        const uint64_t k = k0 + threadIdx.x;
        uint32_t s = 0, at = 0;
        if (k < nitems) {
            s = skey[k];
            at = atomicAdd(&h[s], 1u);
        }
        __syncthreads();
        const uint32_t cnt = h[threadIdx.x];
        const uint32_t base = cnt ? atomicAdd(&cursors[threadIdx.x], cnt) : 0u;
        __syncthreads();
        h[threadIdx.x] = start[threadIdx.x] + base;
        __syncthreads();
        if (k < nitems) {
            const uint32_t eb = first[k], ee = k + 1 < nitems ? first[k + 1] : ne, j = key[eb];
            const uint32_t t0 = rowptr[j], t1 = rowptr[j + 1];
            uint32_t g = 0;
            if (csegs) {
                uint32_t hi = graphs;  // rowptr[csegs[g]] <= t0 < rowptr[csegs[hi]]
                while (hi - g > 1) {
                    const uint32_t mid = (g + hi) >> 1;
                    if (rowptr[csegs[mid]] <= t0) g = mid;
                    else hi = mid;
                }
            }
            const uint32_t r = h[s] + at;
            items[2 * (size_t)r] = make_uint4(t0, t1, eb, ee);
            items[2 * (size_t)r + 1] = make_uint4((uint32_t)col[t0], (uint32_t)col[t1 - 1],
                                                  (uint32_t)min(P[ee] - P[eb], (uint64_t)0xFFFFFFFFu), g);
        }
        __syncthreads();
    }
}

template <class T>
T read_dev(const T* p, hipStream_t s) {
    T h{};
    BTC_HIP(hipMemcpyAsync(&h, p, sizeof(T), hipMemcpyDeviceToHost, s));
    BTC_HIP(hipStreamSynchronize(s));
    return h;
}

}  // namespace

void plan_device(btc_plan_s* p, int64_t chunk, hipStream_t s) {
    btc_graph_s* g = p->g;
    const int32_t n = g->n;
    const int64_t m = g->m;
    const uint32_t* rowptr = g->d_rowptr.p;
    const int32_t* col = g->d_col.p;
    BTC_REQUIRE(m < (int64_t)0xFFFFFFFFLL, BTC_ERR_OVERFLOW, "nnz(L) %lld exceeds 2^32 - 1", (long long)m);

    TmpBuf<uint32_t> erow;
    erow.alloc((size_t)m, s);
    if (m) BTC_LAUNCH(edge_rows_kernel, (int64_t)n * 64, s, rowptr, n, erow.p);

    // dense mask tiles
    TmpBuf<unsigned long long> st;
    st.alloc(8, s);
    BTC_HIP(hipMemsetAsync(st.p, 0, 64, s));
    TmpBuf<uint8_t> dense;
    p->n_dense = 0;
    if (p->tau < 16 * p->K && m > 0) {
        const btc_bitbsr_s* b = plan_bsr(p, s, true);
        TmpBuf<uint32_t> pop, flag, pos;
        pop.alloc(b->nblk, s);
        flag.alloc(b->nblk, s);
        pos.alloc((size_t)b->nblk + 1, s);
        launch_tile_popcount(b, pop.p, s);
        BTC_LAUNCH_RED(dense_tiles_kernel, b->nblk, s, pop.p, b->nblk, p->tau, flag.p, st.p + 0);
        exclusive_scan_u32(flag.p, pos.p, b->nblk, s);
        const uint32_t nd = read_dev(pos.p + b->nblk, s);
        if (nd) {
            p->dense_list.alloc_on(nd, s);
            BTC_LAUNCH(select_kernel, b->nblk, s, flag.p, pos.p, (int64_t)b->nblk, p->dense_list.p);
            dense.alloc((size_t)m, s);
            BTC_LAUNCH(dense_edges_kernel, m, s, col, erow.p, m, p->K, b->indptr.p, b->indices.p, pop.p, p->tau,
                       dense.p);
            p->n_dense = nd;
        }
        BTC_HIP(hipStreamSynchronize(s));
        if (!nd) drop_plan_bsr(p, s);
    }
    p->info.dense_tiles = p->n_dense;
    p->info.dense_edges = (int64_t)read_dev(st.p + 0, s);

    // hub-core bitmaps
    TmpBuf<uint32_t> cend, has, rbi;
    cend.alloc((size_t)n, s);
    has.alloc((size_t)n, s);
    rbi.alloc((size_t)n + 1, s);
    const uint32_t C = p->core_ids;
    if (n) BTC_LAUNCH(core_rows_kernel, n, s, rowptr, col, n, C, cend.p, has.p);
    exclusive_scan_u32(has.p, rbi.p, (size_t)n, s);

    // prefix lists: flag and record, compact (pivot, edge), stable sort by pivot
    TmpBuf<uint4> rec;
    TmpBuf<uint32_t> lflag, lpos;
    rec.alloc((size_t)m, s);
    lflag.alloc((size_t)m, s);
    lpos.alloc((size_t)m + 1, s);
    if (m)
        BTC_LAUNCH_CLIP(clip_kernel, m, s, rowptr, col, erow.p, p->n_dense ? dense.p : nullptr, m, cend.p, has.p, rbi.p, C,
                        lflag.p, rec.p, st.p + 1);
    exclusive_scan_u32(lflag.p, lpos.p, (size_t)m, s);
    const uint32_t nbm = read_dev(rbi.p + n, s);
    const uint32_t ne = read_dev(lpos.p + m, s);
    TmpBuf<uint32_t> k0, v0, k1, v1;
    k0.alloc(ne, s);
    v0.alloc(ne, s);
    k1.alloc(ne, s);
    v1.alloc(ne, s);
    if (m) BTC_LAUNCH(list_keys_kernel, m, s, lflag.p, lpos.p, col, m, k0.p, v0.p);
    lflag.release();
    lpos.release();
    dense.release();
    const bool alt = sort_pairs_u32(k0.p, v0.p, k1.p, v1.p, ne, id_bits(n), s);
    const uint32_t* key = alt ? k1.p : k0.p;
    const uint32_t* val = alt ? v1.p : v0.p;
    // the sort's spare arrays go before the lists come, the prefix sums come
    // after the entries' records have gone: some 56 bytes an entry at the most
    // beside L and the dense tiles
    (alt ? k0 : k1).release();
    (alt ? v0 : v1).release();
    TmpBuf<uint32_t> off;
    off.alloc((size_t)n + 1, s);
    BTC_LAUNCH(pivot_offsets_kernel, (int64_t)n + 1, s, key, ne, n, off.p);

    // one allocation: list records, row bitmaps, list rows; items apart
    const size_t lb = (size_t)ne * sizeof(uint4), bb = (size_t)nbm * (C / 32) * 4, rb = (size_t)ne * 4;
    p->lists.alloc_on(lb + bb + rb, s);
    uint4* lst = reinterpret_cast<uint4*>(p->lists.p);
    uint32_t* rowbits = reinterpret_cast<uint32_t*>(p->lists.p + lb);
    int32_t* ur = reinterpret_cast<int32_t*>(p->lists.p + lb + bb);
    if (bb) {
        BTC_LAUNCH(core_fill_kernel, (int64_t)n * 64, s, rowptr, col, cend.p, has.p, rbi.p, n, C, rowbits);
    }
    TmpBuf<uint64_t> cost, P;
    cost.alloc(ne, s);
    if (ne)
        BTC_LAUNCH_CLIP(records_kernel, ne, s, rowptr, col, erow.p, key, val, (int64_t)ne, rec.p, C, lst, ur, cost.p,
                        st.p + 3, st.p + 6);
    rec.release();
    P.alloc((size_t)ne + 1, s);
    exclusive_scan_u64(cost.p, P.p, ne, s);
    erow.release();

    // work items
    TmpBuf<uint32_t> start, spos;
    start.alloc(ne, s);
    spos.alloc((size_t)ne + 1, s);
    if (ne) BTC_LAUNCH(item_start_kernel, ne, s, rowptr, col, key, off.p, P.p, (int64_t)ne, (uint64_t)chunk, start.p);
    exclusive_scan_u32(start.p, spos.p, ne, s);
    const uint32_t nitems = read_dev(spos.p + ne, s);
    TmpBuf<uint32_t> first, sk0, sv0, sk1, sv1;
    first.alloc(nitems, s);
    if (ne) BTC_LAUNCH(select_kernel, ne, s, start.p, spos.p, (int64_t)ne, first.p);
    TmpBuf<uint4> tmp;
    tmp.alloc((size_t)nitems * 2, s);
    sk0.alloc(nitems, s);
    sv0.alloc(nitems, s);
    sk1.alloc(nitems, s);
    sv1.alloc(nitems, s);
    if (nitems)
        BTC_LAUNCH_RED(items_kernel, nitems, s, rowptr, col, key, off.p, P.p, first.p, nitems, ne,
                   p->use_tiny, p->tiny_all, tmp.p, sk0.p, sv0.p, st.p + 4);
    const bool ialt = sort_pairs_u32(sk0.p, sv0.p, sk1.p, sv1.p, nitems, 32, s);
    p->items_dev.alloc_on((size_t)nitems * 2, s);
    if (nitems)
        BTC_LAUNCH(place_items_kernel, nitems, s, tmp.p, ialt ? sv1.p : sv0.p, nitems, p->items_dev.p);

    // st: [0] dense edges, [1] sparse edges, [2] their merge work, [3] core
    // lists, [4] pivot row words over items, [5] wave items (tiny ones
    // included), [6] ids looked up in the 16-bit copy, [7] tiny items
    unsigned long long h[8];
    BTC_HIP(hipMemcpyAsync(h, st.p, sizeof(h), hipMemcpyDeviceToHost, s));
    const uint64_t checks = read_dev(P.p + ne, s);  // synchronises h as well
    p->items_p = p->items_dev.p;
    p->list_p = lst;
    p->rowbits_p = reinterpret_cast<const uint4*>(rowbits);
    p->urow_p = ur;
    p->nitems = nitems;
    p->n_block_items = nitems - (uint32_t)h[5];
    p->n_tiny_items = (uint32_t)h[7];
    p->info.tiny_items = p->n_tiny_items;
    p->info.sparse_edges = (int64_t)h[1];
    p->info.sparse_merge_work = (int64_t)h[2];
    p->info.core_lists = (int64_t)h[3];
    p->info.core_rows = nbm;
    p->info.wedge_checks = (int64_t)checks;
    p->info.work_items = nitems;
    // looked-up ids (4 B, or 2 B below kNarrowIds), core words and pivot
    // rows (4 B), list records (16 B), items (32 B)
    p->info.stream_bytes = 4 * ((int64_t)checks + (int64_t)h[4]) - 2 * (int64_t)h[6] + 16 * (int64_t)ne +
                           32 * (int64_t)nitems;
}

namespace {

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
        hipLaunchKernelGGL(kernel, dim3(std::min(cap_grid(cap), 4 * kCapRedBlocks)), dim3(kT), 0, s, __VA_ARGS__);  \
        BTC_CHECK_LAUNCH(#kernel);                                                         \
    } while (0)

void plan_capacity(const PlanCap& c, hipStream_t s) {
    PipeCtl* ctl = c.ctl;
    const Cnt nc = Cnt::dev(&ctl->nc);
    const int64_t M = c.m_cap, N = c.n_cap, I = (int64_t)c.items_cap;
    const uint32_t C = c.core_ids;
    const SortUse su = dseq_sort(*c.seq, id_bits(c.n_cap));
    CAP_LAUNCH(pipe_rows_kernel, N, s, c.rowptr, c.col, ctl, C, c.cend, c.rbi);
    if (C) CAP_LAUNCH(core_fill_kernel, N * 64, s, c.rowptr, c.col, c.cend, nullptr, c.rbi, nc, C, c.rowbits);
    with_tile_per(M, [&](auto per) {
        constexpr int PER = decltype(per)::value;
        // prefix lists: records by entry, (pivot, entry) pairs, stably sorted by pivot
        CAP_LAUNCH_RED(pipe_clip_kernel<PER>, M / PER + 1, s, c.rowptr, c.col, c.erow, c.cend, c.rbi, C, ctl, c.k0, c.v0,
                       c.rec, su, dseq_scan(*c.seq));
        const bool alt = dsort_pairs_u32(c.k0, c.v0, c.k1, c.v1, (size_t)M, &ctl->ne, su, s);
        const uint32_t* key = alt ? c.k1 : c.k0;
        const uint32_t* val = alt ? c.v1 : c.v0;
        // records, costs and pivots' ranges in list order
        CAP_LAUNCH_RED(pipe_lists_kernel<PER>, M / PER + 1, s, c.rowptr, c.col, c.erow, C, ctl, key, val, c.rec, c.off,
                       c.oend, c.lists, c.ur, c.P, dseq_scan(*c.seq));
        // work items (each opens at a list, so there are at most ne of them):
        // about 64 per CU, by class and then work in half octaves
        CAP_LAUNCH(pipe_first_kernel<PER>, M / PER + 1, s, c.rowptr, c.col, ctl, key, c.off, c.oend, c.P,
                   (uint64_t)64 * (uint64_t)c.cus, c.first, dseq_scan(*c.seq));
        const SortUse iu = dseq_sort(*c.seq, kDigitBits);  // its words: bucket totals, then cursors
        CAP_LAUNCH_RED(pipe_item_keys_kernel, I, s, c.rowptr, c.col, ctl, key, c.off, c.oend, c.P, c.first, c.skey,
                       iu.totals);
        CAP_LAUNCH_RED(pipe_place_kernel, I, s, c.rowptr, c.col, ctl, key, c.P, c.first, c.skey, iu.totals,
                       iu.totals + kDigits, c.csegs, c.items);
    });
}

}  // namespace btcx
