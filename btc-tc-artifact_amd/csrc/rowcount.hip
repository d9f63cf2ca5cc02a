// Sparse part of the Bit-BSR count: the mask bits of tiles that are not
// dense, evaluated row by row over the CSR of L that a Bit-BSR handle keeps
// beside its tiles.
//
// For a row i with ids N(i), every mask bit (i, j) counts |N(i) & N(j)|.
// A team (16 lanes, a wave or a workgroup, by the row's length) puts N(i)
// into LDS once -- a bitmap window when the row's ids span few enough ids,
// else a table of 4-slot buckets -- and streams the lists N(j) of its mask
// bits through it, spread evenly over the lanes with aligned 16-byte loads.
// The whole sum belongs to vertex i, so per-vertex counts cost one atomic
// per item.
//
// Why not tile by tile: a sparse tile holds one to four bits, so a wave per
// mask tile walks two tile-column lists for one row intersection, most of
// whose matched tile pairs are empty in that row.  Rows read only ids that
// can match.  Count calls on MI355X, a wave per mask tile with per-lane
// merges against rows: Erdos-Renyi 2^14 (131 K edges, 16 x 32) 720 -> 35 us,
// planted 2^17 (4.4 M edges, 16 x 128, dense tiles apart) 939 -> 206 us,
// R-MAT 2^17 in id order (1.9 M edges, 16 x 128, per vertex) 7445 -> 479 us.
// Bound: VALU issue in the membership tests (60 to 75 % of the issue slots
// on the last two), the rest the latency of short rows' load chains.
#include "device_util.h"
#include "internal.h"

namespace btcx {
namespace {

constexpr int kT = 256;
constexpr int kRowWords = 4096;              // LDS words of a workgroup: 16 KiB, so 8 workgroups stay resident per CU
constexpr int kRowWaveWords = kRowWords / 4;  // a wave's slice
constexpr int kRowTeam = 16;                 // lanes of a light row's team
constexpr int kRowTeamWords = kRowWords / (kT / kRowTeam);
constexpr uint32_t kShortQuads = 8;          // 4 lanes in two steps
// A list of more than kSearchLen ids is searched for the row's pc ids below j
// where streaming it takes more than kSearchCost ids per step of the search
// (R-MAT 2^17, kernel: cost 1 / 2 / 4 / 8 444 / 426 / 490 / 511 us, lists
// above 64 / 256 / 1024 / 16000 ids 426 / 441 / 497 / 564 us).
constexpr uint32_t kSearchCost = 2;
constexpr uint32_t kSearchLen = 64;
constexpr uint32_t kEmptySlot = 0xFFFFFFFFu;  // above every id, as kNoId
constexpr uint32_t kNoId = 0xFFFFFFFEu;       // in place of a loaded id that is not the list's

// Rows of at most kLightRow ids go to 16-lane teams (4 per wave, so the
// dependent loads of 4 short rows overlap), rows of at most kWaveRow ids to
// waves in items of kWaveLists lists, longer ones to workgroups in items of
// kBlockLists lists: an item rebuilds its row's set, which costs d / team
// steps against the sum of its lists' ids / (4 team), so the cut keeps an
// item's cost near its neighbours' without the rebuild showing.
constexpr uint32_t kLightRow = 64;   // = the bucket table's load 1/4 in kRowTeamWords
constexpr uint32_t kWaveRow = 512;   // = load 1/2 in kRowWaveWords
constexpr uint32_t kWaveLists = 64;
constexpr uint32_t kBlockLists = 256;

// Item classes of a row of d ids; a row of fewer than two closes no triangle.
__device__ __forceinline__ int row_class(uint32_t d) { return d < 2 ? -1 : d <= kLightRow ? 0 : d <= kWaveRow ? 1 : 2; }

// Items of a row of class k and d ids.
__device__ __forceinline__ uint32_t row_class_items(int k, uint32_t d) {
    return k == 0 ? 1u : k == 1 ? (d + kWaveLists - 1) / kWaveLists : (d + kBlockLists - 1) / kBlockLists;
}

// Copies rowptr and col and lists every row's items {t0, t1, first list,
// row} by class: light at items[0], wave at items[cap0], workgroup at
// items[cap0 + cap1].  count[0..2] = items per class (cleared before).  A
// workgroup takes kItemRows rows at a time and adds each class's items with
// one atomic (one per wave took 52 us of a 262,144-row build, nearly all of
// it the same-address atomics).
constexpr uint32_t kItemRows = 4 * kT;
__global__ __launch_bounds__(kT) void row_items_kernel(const uint32_t* __restrict__ rowptr_in,
                                                       const int32_t* __restrict__ col_in, uint32_t n, uint64_t ncol,
                                                       uint32_t* __restrict__ rowptr, int32_t* __restrict__ col,
                                                       uint4* __restrict__ items, uint64_t cap0, uint64_t cap1,
                                                       uint32_t* __restrict__ count) {
    __shared__ uint32_t wsum[3][kT / 64], base_s[3];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const uint64_t stride = (uint64_t)gridDim.x * kT;
    for (uint64_t q = (uint64_t)blockIdx.x * kT + tid; q < ncol; q += stride) col[q] = col_in[q];
    for (uint64_t base = (uint64_t)blockIdx.x * kItemRows; base <= n; base += (uint64_t)gridDim.x * kItemRows) {
        uint32_t a[4], d[4], sum[3] = {0, 0, 0};
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const uint64_t i = base + x * kT + tid;
            a[x] = d[x] = 0;
            if (i <= n) {
                a[x] = rowptr_in[i];
                rowptr[i] = a[x];
                d[x] = (i < n ? rowptr_in[i + 1] : a[x]) - a[x];
            }
            const int cls = row_class(d[x]);
#pragma unroll
            for (int k = 0; k < 3; ++k) sum[k] += cls == k ? row_class_items(k, d[x]) : 0u;
        }
        uint32_t at[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            uint32_t inc = sum[k];  // inclusive scan over the wave
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t y = (uint32_t)__shfl_up((int)inc, o);
                if ((int)lane >= o) inc += y;
            }
            at[k] = inc - sum[k];
            if (lane == 63) wsum[k][wv] = inc;
        }
        __syncthreads();
        if (tid < 3) {
            const uint32_t t = wsum[tid][0] + wsum[tid][1] + wsum[tid][2] + wsum[tid][3];
            base_s[tid] = t ? atomicAdd(&count[tid], t) : 0u;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            at[k] += base_s[k];
            for (uint32_t w = 0; w < wv; ++w) at[k] += wsum[k][w];
        }
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const uint64_t i = base + x * kT + tid;
            const int cls = row_class(d[x]);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                if (cls != k) continue;
                uint4* out = items + (k == 0 ? 0 : k == 1 ? cap0 : cap0 + cap1);
                const uint32_t per = k == 1 ? kWaveLists : kBlockLists, c = row_class_items(k, d[x]);
                for (uint32_t y = 0; y < c; ++y) out[at[k]++] = make_uint4(a[x], a[x] + d[x], a[x] + y * per, (uint32_t)i);
            }
        }
        __syncthreads();  // the next rows rewrite the sums
    }
}

// Barrier of the threads that share an item's LDS.
template <int NT>
__device__ __forceinline__ void row_sync() {
    if constexpr (NT == kT) {
        __syncthreads();
    } else {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// 1 when k is among the ascending ids col[lo, hi).
__device__ __forceinline__ uint32_t sorted_has(const int32_t* __restrict__ col, uint32_t lo, uint32_t hi, uint32_t k) {
    const uint32_t end = hi;
    while (lo < hi) {
        const uint32_t mid = lo + ((hi - lo) >> 1);
        if ((uint32_t)col[mid] < k) lo = mid + 1;
        else hi = mid;
    }
    return lo < end && (uint32_t)col[lo] == k ? 1u : 0u;
}

// Sets over N(i) in W words of LDS.
// Bitmap: bit k - base; ids outside the window land on its last bit, which
// is never set.
template <int W>
struct RowBitmap {
    const uint32_t* w;
    uint32_t base;
    __device__ __forceinline__ uint32_t has(uint32_t k) const {
        const uint32_t x = min(k - base, 32u * W - 1u);
        return (w[x >> 5] >> (x & 31u)) & 1u;
    }
    __device__ __forceinline__ uint32_t has4(uint4 k) const { return has(k.x) + has(k.y) + has(k.z) + has(k.w); }
};

// W / 4 buckets of 4 ids, one 16-byte read per test; a full bucket spills
// into the next one.  At load 1/4 (light rows) one bucket in 270 is full, so
// nearly every test is one LDS read, where linear probing loops until the
// slowest of 64 lanes meets an empty slot.
template <int W>
struct RowBuckets {
    uint32_t* w;
    __device__ __forceinline__ static uint32_t bucket(uint32_t k) {
        return (k * 2654435761u) >> (32 - __builtin_ctz((unsigned)W / 4));
    }
    __device__ __forceinline__ void insert(uint32_t k) const {
        uint32_t b = bucket(k);
        for (;;) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
                if (atomicCAS(&w[4 * b + s], kEmptySlot, k) == kEmptySlot) return;
            b = (b + 1) & (W / 4 - 1);
        }
    }
    __device__ __forceinline__ uint4 read(uint32_t b) const { return *reinterpret_cast<const uint4*>(w + 4 * b); }
    __device__ __forceinline__ static bool match(uint4 v, uint32_t k) {
        return v.x == k || v.y == k || v.z == k || v.w == k;
    }
    // slots of a bucket fill in order, so an empty last slot ends the chain
    __device__ uint32_t has_past(uint32_t b, uint32_t k) const {
        for (;;) {
            b = (b + 1) & (W / 4 - 1);
            const uint4 v = read(b);
            if (match(v, k)) return 1u;
            if (v.w == kEmptySlot) return 0u;
        }
    }
    // the four first buckets are read together
    __device__ __forceinline__ uint32_t has4(uint4 k) const {
        const uint32_t b0 = bucket(k.x), b1 = bucket(k.y), b2 = bucket(k.z), b3 = bucket(k.w);
        const uint4 v0 = read(b0), v1 = read(b1), v2 = read(b2), v3 = read(b3);
        const bool m0 = match(v0, k.x), m1 = match(v1, k.y), m2 = match(v2, k.z), m3 = match(v3, k.w);
        uint32_t h = (uint32_t)m0 + (uint32_t)m1 + (uint32_t)m2 + (uint32_t)m3;
        if (!m0 && v0.w != kEmptySlot) h += has_past(b0, k.x);
        if (!m1 && v1.w != kEmptySlot) h += has_past(b1, k.y);
        if (!m2 && v2.w != kEmptySlot) h += has_past(b2, k.z);
        if (!m3 && v3.w != kEmptySlot) h += has_past(b3, k.w);
        return h;
    }
};

// Spreads the units of the lanes' lists (units[x] of lane x, 0 = none) over
// the wave, 64 at a time in list order: f(active, lane x's a, b, c, unit
// index within the list).  Lists of a wave differ in length by orders of
// magnitude, and a fixed set of lanes per list runs as long as its longest
// one; this way every step has 64 busy lanes.  The lane that a unit belongs
// to comes from a 64-bit mask of list starts kept in scalar registers.
// Wave-uniform call; the units of one call sum to less than 2^32.
template <class F>
__device__ __forceinline__ void spread_units(uint32_t units, uint32_t a, uint32_t b, uint32_t c, int lane, F&& f) {
    const uint64_t some = __ballot(units != 0);
    if (!some) return;
    const uint32_t cnt = (uint32_t)__popcll(some);
    const uint64_t below = (1ull << lane) - 1;
    // lists with units first, order kept (a permutation of the lanes)
    const uint32_t to = units ? (uint32_t)__popcll(some & below) : cnt + (uint32_t)__popcll(~some & below);
    units = (uint32_t)__builtin_amdgcn_ds_permute((int)(4 * to), (int)units);
    a = (uint32_t)__builtin_amdgcn_ds_permute((int)(4 * to), (int)a);
    b = (uint32_t)__builtin_amdgcn_ds_permute((int)(4 * to), (int)b);
    c = (uint32_t)__builtin_amdgcn_ds_permute((int)(4 * to), (int)c);
    uint32_t start = units;  // exclusive prefix
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)start, o);
        if (lane >= o) start += y;
    }
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)start, 63);
    start -= units;
    uint32_t next = 0, next_at = 0;  // the next list to start, and where
    for (uint32_t t0 = 0; t0 < total; t0 += 64) {
        uint64_t m = 0;
        const uint32_t first = next;
        while (next < cnt && next_at < t0 + 64) {
            m |= 1ull << (next_at - t0);
            ++next;
            next_at = (uint32_t)__builtin_amdgcn_readlane((int)start, (int)min(next, 63u));
        }
        const uint32_t x = first + (uint32_t)__popcll(m & (below | (1ull << lane))) - 1;
        const uint32_t t = t0 + (uint32_t)lane;
        f(t < total, (uint32_t)__shfl((int)a, (int)x), (uint32_t)__shfl((int)b, (int)x),
          (uint32_t)__shfl((int)c, (int)x), t - (uint32_t)__shfl((int)start, (int)x));
    }
}

struct RowsArgs {
    const uint32_t* rowptr;
    const int32_t* col;
    const uint16_t* epop;  // set: entries in tiles of more than tau bits are left out
    int tau;
    const uint4* items[3];  // light, wave, workgroup
    uint32_t count[3];
    unsigned long long* slots;
    PvOut pv;
};

// The rows of a wave's current items: TN sets side by side in LDS (TN = 4
// light rows, else 1).  Uniform over the wave.
template <int TN>
struct WaveRows {
    uint32_t t0[TN];        // first entry of the row
    uint32_t e0[TN];        // first list taken
    uint32_t upto[TN + 1];  // lists of rows below r: upto[r]
};

// The lists of a wave's rows: list e of row r is N(j), j = col[e].  64 lists
// at a time get their bounds, a lane each, two rounds ahead (the ids) and
// one round ahead (the bounds) of the round being scanned: a round of short
// lists is otherwise a chain of three dependent loads.  The first bounds are
// asked for before the sets are built.  Rounds start at c0, step cs; lane x
// takes list c + x LS of a round, so that the waves of a workgroup (LS = 4, c0
// = wave) share the long lists at a row's end.
template <int TN, uint32_t LS>
struct ListFeed {
    const RowsArgs& a;
    const WaveRows<TN>& w;
    const uint32_t lane, cs;
    uint32_t c;         // current round's first list
    uint32_t r0, r1;    // bounds of this lane's list (0, 0: none)
    uint32_t next_j;    // id of its list of the next round (kEmptySlot: none)

    // row of list g, its entry of L and the row's first one
    __device__ __forceinline__ void place(uint32_t g, uint32_t& r, uint32_t& e, uint32_t& t0) const {
        r = 0;
        e = w.e0[0] + g;
        t0 = w.t0[0];
#pragma unroll
        for (int k = 1; k < TN; ++k)
            if (g >= w.upto[k]) {
                r = (uint32_t)k;
                e = w.e0[k] + (g - w.upto[k]);
                t0 = w.t0[k];
            }
    }
    __device__ __forceinline__ uint32_t id(uint32_t at) const {
        const uint32_t g = at + lane * LS;
        uint32_t r, e, t0, j = kEmptySlot;
        place(g, r, e, t0);
        // nothing of the row lies below its first id
        if (g < w.upto[TN] && e != t0) {
            j = (uint32_t)a.col[e];
            if (a.epop && (int)a.epop[e] > a.tau) j = kEmptySlot;
        }
        return j;
    }
    __device__ __forceinline__ void bounds(uint32_t j, uint32_t& b0, uint32_t& b1) const {
        b0 = b1 = 0;
        if (j != kEmptySlot) {
            b0 = a.rowptr[j];
            b1 = a.rowptr[j + 1];
        }
    }
    __device__ __forceinline__ ListFeed(const RowsArgs& a_, const WaveRows<TN>& w_, uint32_t lane_, uint32_t c0,
                                        uint32_t cs_)
        : a(a_), w(w_), lane(lane_), cs(cs_), c(c0) {
        const uint32_t j = id(c);
        next_j = id(c + cs);
        bounds(j, r0, r1);
    }
};

// Whether a list of len ids is searched for the pc ids of the row below it.
__device__ __forceinline__ bool searched(uint32_t len, uint32_t pc) {
    return len > kSearchLen && (uint64_t)len > (uint64_t)pc * kSearchCost * (uint32_t)(32 - __clz((int)len));
}

// Aligned quads that hold col[r0, r1).
__device__ __forceinline__ uint32_t list_quads(uint32_t r0, uint32_t r1) {
    return r0 < r1 ? (r1 - (r0 & ~3u) + 3) / 4 : 0u;
}

// Quad u of the list of n ids at a0 (col is padded past its end): ids before
// the list (o wraps) or past it become kNoId, which no set holds.
__device__ __forceinline__ uint4 list_quad(const int32_t* __restrict__ col, uint32_t a0, uint32_t n, uint32_t u) {
    uint4 v = *reinterpret_cast<const uint4*>(col + (a0 & ~3u) + (size_t)u * 4);
    const uint32_t o = 4 * u - (a0 & 3u);
    v.x = o + 0 < n ? v.x : kNoId;
    v.y = o + 1 < n ? v.y : kNoId;
    v.z = o + 2 < n ? v.z : kNoId;
    v.w = o + 3 < n ? v.w : kNoId;
    return v;
}

// Scans the lists of a feed: set(r) gives row r's set, the lists' ids stream
// through the sets, 4 per lane and step.  Only the row's ids below j can
// match in N(j): where they are so few that searching them in a long list
// takes less, that list is searched instead.  hits(r, h) collects h hits of
// row r.
template <int TN, uint32_t LS, class SetOf, class Hits>
__device__ __forceinline__ void scan_wave(ListFeed<TN, LS>& f, SetOf&& set, Hits&& hits) {
    const RowsArgs& a = f.a;
    const int lane = (int)f.lane;
    while (f.c < f.w.upto[TN]) {
        uint32_t n0, n1;
        f.bounds(f.next_j, n0, n1);
        f.next_j = f.id(f.c + 2 * f.cs);
        uint32_t r, e, t0;
        f.place(f.c + f.lane * LS, r, e, t0);
        const uint32_t r0 = f.r0, len = f.r1 - f.r0, pc = e - t0;
        const bool search = searched(len, pc);
        const uint32_t quads = search ? 0u : list_quads(r0, f.r1);
        auto quad = [&](bool on, uint32_t a0, uint32_t n, uint32_t row, uint32_t u) {
            const auto st = set(row);  // reads other lanes
            hits(row, on ? st.has4(list_quad(a.col, a0, n, u)) : 0u);
        };
        if (__any(quads > kShortQuads)) {
            spread_units(quads, r0, len, r, lane, quad);
        } else {
            // short lists only: 4 lanes each, 16 lists a step
#pragma unroll 1
            for (int s = 0; s < 4; ++s) {
                const int x = s * 16 + lane / 4;
                const uint32_t nq = (uint32_t)__shfl((int)quads, x);
                if (!__any(nq != 0)) continue;
                const uint32_t a0 = (uint32_t)__shfl((int)r0, x), n = (uint32_t)__shfl((int)len, x),
                               row = TN > 1 ? (uint32_t)__shfl((int)r, x) : 0u, u = (uint32_t)lane & 3u;
                quad(u < nq, a0, n, row, u);
                if (__any(nq > 4)) quad(u + 4 < nq, a0, n, row, u + 4);
            }
        }
        spread_units(search ? pc : 0u, r0, len, TN > 1 ? r : 0u, lane,
                     [&](bool on, uint32_t a0, uint32_t n, uint32_t row, uint32_t u) {
                         uint32_t h = 0, first = f.w.t0[0];
#pragma unroll
                         for (int k = 1; k < TN; ++k) first = row == (uint32_t)k ? f.w.t0[k] : first;
                         if (on) h = sorted_has(a.col, a0, a0 + n, (uint32_t)a.col[first + u]);
                         hits(row, h);
                     });
        f.r0 = n0;
        f.r1 = n1;
        f.c += f.cs;
    }
}

// One row's set in LDS by NT threads (rank tid): its ids [t0, t0 + d).
template <int NT, int W>
__device__ __forceinline__ void build_window(const int32_t* __restrict__ col, uint32_t t0, uint32_t d, uint32_t base,
                                             uint32_t hi, uint32_t* lds, uint32_t tid) {
    const uint32_t nw = ((hi - base) >> 5) + 1u;
    for (uint32_t w = 4 * tid; w < nw; w += 4 * NT) *reinterpret_cast<uint4*>(lds + w) = make_uint4(0, 0, 0, 0);
    if (tid == 0) lds[W - 1] = 0;  // ids outside [base, hi]; list ids inside are below hi, so in the cleared words
    row_sync<NT>();
    for (uint32_t x = tid; x < d; x += NT) {
        const uint32_t k = (uint32_t)col[t0 + x] - base;
        atomicOr(&lds[k >> 5], 1u << (k & 31u));
    }
    row_sync<NT>();
}

template <int NT, int W>
__device__ __forceinline__ void build_buckets(const int32_t* __restrict__ col, uint32_t t0, uint32_t d, uint32_t* lds,
                                              uint32_t tid) {
    for (uint32_t w = 4 * tid; w < (uint32_t)W; w += 4 * NT)
        *reinterpret_cast<uint4*>(lds + w) = make_uint4(kEmptySlot, kEmptySlot, kEmptySlot, kEmptySlot);
    row_sync<NT>();
    const RowBuckets<W> set{lds};
    for (uint32_t x = tid; x < d; x += NT) set.insert((uint32_t)col[t0 + x]);
    row_sync<NT>();
}

// Lists of a row that fits neither LDS set (more than half the table's slots
// over a span beyond the bitmap's), by a workgroup: windows of the id space one
// after the other, each with the bitmap of the row's ids in it, and of every
// list the part in the window.  `f` holds a wave's lists, at most 64.  Lists
// that are searched take no window.  Bound: one workgroup a row's item, and
// where the last few lists are long that is all a row has (60 rows of 100 K
// ids over 3 M: count 2.9 ms; this kernel alone 83 with a search of the row for
// every id).
template <int W, uint32_t LS, class Hits>
__device__ __forceinline__ void scan_windows(ListFeed<1, LS>& f, uint32_t t1, uint32_t lo, uint32_t hi, uint32_t* lds,
                                             uint32_t tid, Hits&& hits) {
    // the last word stays empty: ids outside the window (kNoId) land there
    constexpr uint32_t kSpan = 32u * (W - 1);
    const RowsArgs& a = f.a;
    const int lane = (int)f.lane;
    uint32_t r, e, t0;
    f.place(f.c + f.lane * LS, r, e, t0);
    const uint32_t first = f.w.t0[0], r0 = f.r0, r1 = f.r1, pc = e - t0;
    const bool search = searched(r1 - r0, pc);
    spread_units(search ? pc : 0u, r0, r1 - r0, 0u, lane, [&](bool on, uint32_t a0, uint32_t n, uint32_t, uint32_t u) {
        hits(0u, on ? sorted_has(a.col, a0, a0 + n, (uint32_t)a.col[first + u]) : 0u);
    });
    uint32_t p = search ? r1 : r0;  // the list's ids from here on are still to come
    uint32_t at = first;            // the row's
    uint32_t base = lo & ~31u;
    while (__syncthreads_or(p < r1)) {
        const uint32_t end = base + kSpan;  // below 2^32: ids are below 2^31
        for (uint32_t w = 4 * tid; w < (uint32_t)W; w += 4 * kT)
            *reinterpret_cast<uint4*>(lds + w) = make_uint4(0, 0, 0, 0);
        __syncthreads();
        for (;;) {
            const uint32_t k = (uint64_t)at + tid < t1 ? (uint32_t)a.col[at + tid] : 0xFFFFFFFFu;
            if (k < end) atomicOr(&lds[(k - base) >> 5], 1u << ((k - base) & 31u));
            const uint32_t in = (uint32_t)__syncthreads_count(k < end);
            at += in;
            if (in < (uint32_t)kT) break;
        }
        __syncthreads();
        uint32_t z = p, zh = r1;  // first id of the list at or past the window's end
        while (z < zh) {
            const uint32_t mid = z + ((zh - z) >> 1);
            if ((uint32_t)a.col[mid] < end) z = mid + 1;
            else zh = mid;
        }
        const RowBitmap<W> set{lds, base};
        spread_units(list_quads(p, z), p, z - p, 0u, lane, [&](bool on, uint32_t a0, uint32_t n, uint32_t, uint32_t u) {
            hits(0u, on ? set.has4(list_quad(a.col, a0, n, u)) : 0u);
        });
        p = z;
        __syncthreads();  // the next window rewrites the bitmap
        if (end > hi) break;  // workgroup-uniform; list ids are below hi
        base = end;
    }
}

// Lists [it.z, ee) of one row by a wave (NT = 64) or a workgroup.
template <int NT, int W, bool PV>
__device__ __forceinline__ uint64_t row_item(const RowsArgs& a, uint4 it, uint32_t ee, uint32_t* lds, uint32_t tid) {
    const uint32_t t0 = uniform(it.x), d = uniform(it.y) - t0;
    const uint32_t lo = uniform((uint32_t)a.col[t0]), hi = uniform((uint32_t)a.col[t0 + d - 1]);
    const uint32_t base = lo & ~31u;
    const WaveRows<1> w{{t0}, {uniform(it.z)}, {0u, uniform(ee) - uniform(it.z)}};
    constexpr uint32_t LS = NT / 64;
    ListFeed<1, LS> feed(a, w, tid & 63, NT == kT ? uniform(tid / 64) : 0u, NT);
    uint32_t mine = 0;
    auto add = [&](uint32_t, uint32_t h) { mine += h; };
    // Where dense tiles are left out, whole items have no list to scan (most
    // of 12 K items of a complete graph of 2500 ids: kernel 376 -> 282 us with
    // 16 x 128 tiles of more than 512 bits left out).  The answer waits for the
    // lists' bounds, so other counts do not ask.
    static_assert(kBlockLists <= kT && kWaveLists <= 64, "the first round holds every list");
    bool none = false;
    if (a.epop) {
        const bool some = feed.r0 < feed.r1;
        none = NT == kT ? !__syncthreads_or(some) : !__any(some);
    }
    if (none) {
    } else if (hi - base < 32u * W - 1u) {
        build_window<NT, W>(a.col, t0, d, base, hi, lds, tid);
        scan_wave(feed, [&](uint32_t) { return RowBitmap<W>{lds, base}; }, add);
    } else if (NT < kT || d <= (uint32_t)W / 2) {
        build_buckets<NT, W>(a.col, t0, d, lds, tid);
        scan_wave(feed, [&](uint32_t) { return RowBuckets<W>{lds}; }, add);
    } else if constexpr (NT == kT) {
        scan_windows<W>(feed, t0 + d, lo, hi, lds, tid, add);
    }
    row_sync<NT>();  // the next item rewrites the set
    if constexpr (PV) {
        const uint64_t x = wave_sum_u64(mine);
        if ((tid & 63) == 0 && x) pv_add(a.pv, (int64_t)it.w, x);
    }
    return mine;
}

// Four light rows by a wave: lanes 16r..16r+15 build row r's set, all 64
// scan the rows' lists together.  An idle row has no entries.
template <bool PV>
__device__ __forceinline__ uint64_t light_rows(const RowsArgs& a, uint4 it, uint32_t* lds, uint32_t* sums, int lane) {
    constexpr int W = kRowTeamWords;
    const uint32_t t0 = it.x, d = it.y - it.x, r = (uint32_t)lane / kRowTeam, tl = (uint32_t)lane % kRowTeam;
    uint32_t lo = 0, hi = 0;
    if (d) {
        lo = (uint32_t)a.col[t0];
        hi = (uint32_t)a.col[t0 + d - 1];
    }
    const uint32_t base = lo & ~31u;
    WaveRows<4> w;
    w.upto[0] = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        w.t0[k] = w.e0[k] = (uint32_t)__builtin_amdgcn_readlane((int)t0, k * kRowTeam);
        w.upto[k + 1] = w.upto[k] + (uint32_t)__builtin_amdgcn_readlane((int)d, k * kRowTeam);
    }
    ListFeed<4, 1> feed(a, w, (uint32_t)lane, 0u, 64u);
    uint32_t all = 0;
    auto add = [&](uint32_t row, uint32_t h) {
        if constexpr (PV) {
            if (h) atomicAdd(&sums[row], h);
        } else {
            all += h;
        }
    };
    if (PV && lane < 4) sums[lane] = 0;
    if (__all(hi - base < 32u * W - 1u)) {  // one form per wave
        build_window<kRowTeam, W>(a.col, t0, d, base, hi, lds + r * W, tl);
        scan_wave(feed,
                  [&](uint32_t row) {
                      return RowBitmap<W>{lds + row * W, (uint32_t)__shfl((int)base, (int)(row * kRowTeam))};
                  },
                  add);
    } else {
        build_buckets<kRowTeam, W>(a.col, t0, d, lds + r * W, tl);
        scan_wave(feed, [&](uint32_t row) { return RowBuckets<W>{lds + row * W}; }, add);
    }
    row_sync<64>();  // the next rows rewrite the sets
    if constexpr (PV) {
        if (tl == 0) {
            const uint32_t x = sums[r];
            if (x) pv_add(a.pv, (int64_t)it.w, x);
            all = x;
        }
        row_sync<64>();
    }
    return all;
}

// Persistent grid, heaviest class first: workgroup items, wave items, light
// rows (static stride each).  Held to 64 VGPRs: 8 waves per SIMD with a few
// spills against 7, 6 and 5 without (R-MAT 2^17 411 against 503 / 465 / 495
// us, planted 2^17 107 against 125 / 123 / 135 us).
template <bool PV>
__global__ __launch_bounds__(kT, 8) void rows_kernel(RowsArgs a) {
    __shared__ __align__(16) uint32_t lds[kRowWords];
    __shared__ uint32_t sums[kT / kRowTeam];
    __shared__ unsigned long long part[kT / 64];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wv = uniform(tid >> 6);
    uint64_t acc = 0;
    for (uint32_t k = blockIdx.x; k < a.count[2]; k += gridDim.x) {
        const uint4 it = a.items[2][k];
        acc += row_item<kT, kRowWords, PV>(a, it, min(it.y, it.z + kBlockLists), lds, tid);
    }
    // the last workgroup item's closing barrier orders the slices' reuse
    for (uint32_t k = blockIdx.x * 4 + wv; k < a.count[1]; k += gridDim.x * 4) {
        const uint4 it = a.items[1][k];
        acc += row_item<64, kRowWaveWords, PV>(a, it, min(it.y, it.z + kWaveLists), lds + wv * kRowWaveWords, lane);
    }
    constexpr uint32_t TW = 64 / kRowTeam;  // light rows of a wave
    auto light = [&](uint64_t k) {
        const uint64_t mine = k + lane / kRowTeam;
        return mine < a.count[0] ? a.items[0][mine] : make_uint4(0, 0, 0, 0);
    };
    const uint32_t lstep = gridDim.x * 4 * TW;
    uint64_t k = (uint64_t)(blockIdx.x * 4 + wv) * TW;
    uint4 nx = light(k);
    for (; k < a.count[0]; k += lstep) {
        const uint4 it = nx;
        nx = light(k + lstep);
        acc += light_rows<PV>(a, it, lds + wv * kRowWaveWords, sums + wv * TW, (int)lane);
    }
    const uint64_t s = wave_sum_u64(acc);
    if (lane == 0) part[wv] = s;
    __syncthreads();
    if (tid == 0) {
        const unsigned long long x = part[0] + part[1] + part[2] + part[3];
        if (x) atomicAdd(a.slots + kSlotStride * (blockIdx.x % kSlots), x);
    }
}

}  // namespace

void alloc_row_lists(const btc_graph_s* g, RowLists& r, hipStream_t s) {
    const size_t n = (size_t)g->n, m = (size_t)g->m;
    r.m = (int64_t)m;
    r.merge_work = g->merge_work;
    // items: a light row has 2 ids at least; every wave or workgroup item
    // but its row's last holds kWaveLists / kBlockLists lists
    const uint64_t cap0 = std::min<uint64_t>(n, m / 2) + 1;
    const uint64_t cap1 = m / kWaveLists + m / kLightRow + 1;
    const uint64_t cap2 = m / kBlockLists + m / kWaveRow + 1;
    r.cap0 = cap0;
    r.cap1 = cap1;
    const size_t ib = (size_t)(cap0 + cap1 + cap2) * sizeof(uint4);
    const size_t rb = ((n + 1) * 4 + 255) & ~size_t(255);
    r.block.alloc_on(ib + rb + (m + kColPad) * 4 + 4 * RowLists::kCounts + m * 2, s);
    r.items = reinterpret_cast<uint4*>(r.block.p);
    r.rowptr = reinterpret_cast<uint32_t*>(r.block.p + ib);
    r.col = reinterpret_cast<int32_t*>(r.block.p + ib + rb);
    r.d_count = reinterpret_cast<uint32_t*>(r.col + m + kColPad);
    r.epop = reinterpret_cast<uint16_t*>(r.d_count + RowLists::kCounts);
    BTC_HIP(hipMemsetAsync(r.d_count, 0, 4 * RowLists::kCounts, s));
}

void build_row_lists(const btc_graph_s* g, RowLists& r, hipStream_t s) {
    const size_t n = (size_t)g->n, m = (size_t)g->m;
    const size_t work = std::max(n + 1, m + kColPad);
    const unsigned grid = (unsigned)std::min<size_t>((work + kT - 1) / kT, 2048);
    hipLaunchKernelGGL(row_items_kernel, dim3(grid), dim3(kT), 0, s, g->d_rowptr.p, g->d_col.p, (uint32_t)n,
                       (uint64_t)(m + kColPad), r.rowptr, r.col, r.items, r.cap0, r.cap1, r.d_count);
    BTC_CHECK_LAUNCH("row_items_kernel");
}

void launch_rows(const RowLists& r, int tau, unsigned long long* d_slots, PvOut pv, hipStream_t s) {
    const uint64_t waves = (uint64_t)r.count[0] / (64 / kRowTeam) + r.count[1] + 1;
    const uint64_t want = std::max<uint64_t>((waves + 3) / 4, r.count[2]);
    if (r.count[0] == 0 && r.count[1] == 0 && r.count[2] == 0) return;
    const unsigned grid = (unsigned)std::min<uint64_t>(want, (uint64_t)device_cu_count() * 8);
    const bool dense = r.count[3] > (uint32_t)tau;
    RowsArgs a{r.rowptr, r.col, dense ? r.epop : nullptr, tau, {r.items, r.items + r.cap0, r.items + r.cap0 + r.cap1},
               {r.count[0], r.count[1], r.count[2]}, d_slots, pv};
    if (pv.on()) hipLaunchKernelGGL(rows_kernel<true>, dim3(grid), dim3(kT), 0, s, a);
    else hipLaunchKernelGGL(rows_kernel<false>, dim3(grid), dim3(kT), 0, s, a);
    BTC_CHECK_LAUNCH("rows_kernel");
}

}  // namespace btcx
