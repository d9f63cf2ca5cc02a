// Tiles taken in ticket order by the workgroups of one launch, with offsets
// by decoupled look-back, and the digit histograms of the radix sort: the
// parts that the captured build's kernels share with devprim.hip.
//
// Every look-back waits only on tiles whose tickets were taken by running
// workgroups, which publish before they wait, so every wait ends (a spin
// limit sets an error word rather than waiting on).
//
// What bounds these kernels on small inputs is round trips to memory: a
// kernel of a captured graph takes 4 us whatever it does, and atomics on one
// address serialise at some 15 ns each over the eight XCDs.  So steps are
// fused around one tile pass, a workgroup beyond the live tiles leaves
// without a ticket, a grid that covers all tiles takes one ticket per
// workgroup, and nothing counts finished workgroups: tickets, totals and
// statuses are per use and the run's first kernel clears them (prim.h).
#pragma once

#include <type_traits>

#include "device_util.h"
#include "prim.h"

namespace btcx {

constexpr int kTileThreads = 256;

// Look-back status of a tile (and digit): flag << 62 | value; flag 1 = the
// tile's own value, 2 = inclusive of every earlier tile.  Values stay below
// 2^62 (element counts are u32; scanned u64 values are check counts).
constexpr uint64_t kTileAgg = 1ull << 62, kTileInc = 2ull << 62, kTileMask = (1ull << 62) - 1;
constexpr uint32_t kTileSpinMax = 1u << 22;

__device__ __forceinline__ uint64_t tile_load(const uint64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void tile_store(uint64_t* p, uint64_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Waits until the cell at `at`, last read as x, holds a value; past the spin
// limit an inclusive 0, with the error word set.
__device__ __forceinline__ uint64_t tile_settle(const uint64_t* at, uint64_t x, uint32_t* err) {
    for (uint32_t spin = 0; (x >> 62) == 0 && spin < kTileSpinMax; ++spin) {
        __builtin_amdgcn_s_sleep(1);
        x = tile_load(at);
    }
    if ((x >> 62) == 0) {
        atomicOr(err, 1u);
        return kTileInc;
    }
    return x;
}

// Sum of the values of tiles [0, t), by one wave: 64 tiles a round trip, back
// to the nearest inclusive one.  Every lane gets the sum.
__device__ __forceinline__ uint64_t tile_look_back(const uint64_t* cells, uint32_t t, uint32_t* err) {
    const int64_t lane = threadIdx.x & 63;
    uint64_t excl = 0;
    for (int64_t j = (int64_t)t - 1; j >= 0; j -= 64) {
        uint64_t x = kTileInc;  // before the first tile: an inclusive 0
        if (j >= lane) x = tile_settle(cells + (j - lane), tile_load(cells + (j - lane)), err);
        const uint64_t inc = __ballot((x >> 62) == 2);
        const int first = inc ? __builtin_ctzll(inc) : 63;
        excl += wave_sum_u64(lane <= first ? x & kTileMask : 0);
        if (inc) break;
    }
    return excl;
}

// One use of the scan: its ticket, its tiles' statuses and the error word.
struct ScanUse {
    uint32_t* ticket;
    uint64_t* status;
    uint32_t* err;
};

// The tiles of a launch: for (TileLoop l(use, nt); l.next();) with tile l.t.
// Every thread calls next(), which holds barriers.
struct TileLoop {
    uint32_t* ticket;
    uint32_t nt, t;
    bool more;
    uint32_t* s_tile;
    __device__ __forceinline__ TileLoop(uint32_t* ticket_, uint32_t nt_, uint32_t* s_tile_)
        : ticket(ticket_), nt(nt_), t(0), more(blockIdx.x < nt_), s_tile(s_tile_) {}
    __device__ __forceinline__ bool next() {
        if (!more) return false;
        __syncthreads();  // the last tile's readers of *s_tile are through
        if (threadIdx.x == 0) *s_tile = atomicAdd(ticket, 1u);
        __syncthreads();
        t = *s_tile;
        more = gridDim.x < nt;  // else one ticket each covers every tile
        return t < nt;
    }
};

// Exclusive offsets of v[k] over a tile whose element (k, thread) comes at
// k * 256 + thread, added to the sum of all earlier tiles; the tile's own
// sum through the look-back to later ones.  Returns the inclusive total up
// to this tile (thread 0 only).  lds: 4 * PER + 2 values.
template <class T, int PER>
__device__ __forceinline__ uint64_t tile_offsets(const T (&v)[PER], T (&off)[PER], T* lds, const ScanUse& u,
                                                 uint32_t t) {
    static_assert(4 * PER <= 64, "one wave scans the row sums");
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        T x = v[k];
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const T y = __shfl_up(x, o);
            if (lane >= o) x += y;
        }
        off[k] = x - v[k];
        if (lane == 63) lds[k * 4 + wid] = x;
    }
    __syncthreads();
    if (wid == 0) {
        const T own = lane < 4 * PER ? lds[lane] : T(0);
        T x = own;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const T y = __shfl_up(x, o);
            if (lane >= o) x += y;
        }
        if (lane < 4 * PER) lds[lane] = x - own;
        const T tot = __shfl(x, 63);
        uint64_t excl = 0;
        if (t != 0) {
            if (lane == 0) tile_store(u.status + t, kTileAgg | (uint64_t)tot);
            excl = tile_look_back(u.status, t, u.err);
        }
        if (lane == 0) {
            tile_store(u.status + t, kTileInc | (excl + (uint64_t)tot));
            lds[4 * PER] = (T)excl;
            lds[4 * PER + 1] = tot;
        }
    }
    __syncthreads();
    const T excl = lds[4 * PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) off[k] += excl + lds[k * 4 + wid];
    return (uint64_t)excl + (uint64_t)lds[4 * PER + 1];
}

// Elements per thread of a tile pass over up to cap elements: small tiles
// keep 256 CUs busy on small inputs (131 K elements: 256 tiles), large ones
// keep the tickets' serial atomics short beside the data (4 M elements: 2048
// tickets, some 30 us spread over the pass).
template <class F>
inline void with_tile_per(int64_t cap, F&& f) {
    if (cap <= (int64_t(1) << 18)) f(std::integral_constant<int, 2>{});
    else f(std::integral_constant<int, 8>{});
}

// ------------------------------------------------------------ radix digits
constexpr int kDigitBits = 8;
constexpr uint32_t kDigits = 1u << kDigitBits;
constexpr int kMaxPasses = 8;
static_assert(kDigits == (uint32_t)kTileThreads, "one digit per thread");

template <class K>
__device__ __forceinline__ uint32_t digit_of(K k, int shift) {
    return (uint32_t)(k >> shift) & (kDigits - 1);
}

// One use of the sort: what the kernel that writes its keys fills in beside
// them (the digit totals of every pass; the look-back statuses of the live
// tiles cleared), and the passes' tickets.
struct SortUse {
    uint32_t* tickets;   // kMaxPasses
    uint32_t* totals;    // kMaxPasses x kDigits, cleared with the tickets
    uint64_t* status;    // per pass: status_pass words, kDigits per tile
    size_t status_pass;
    uint32_t* err;
    int passes;
    uint32_t tile;       // keys per tile
};

typedef uint32_t DigitHist[kMaxPasses][kDigits];  // __shared__

__device__ __forceinline__ void hist_clear(DigitHist& h, int passes) {
    for (int p = 0; p < passes; ++p) h[p][threadIdx.x] = 0;
    __syncthreads();
}

template <class K>
__device__ __forceinline__ void hist_add(DigitHist& h, int passes, K k) {
    for (int p = 0; p < passes; ++p) atomicAdd(&h[p][digit_of(k, p * kDigitBits)], 1u);
}

__device__ __forceinline__ void hist_flush(DigitHist& h, const SortUse& u) {
    __syncthreads();
    for (int p = 0; p < u.passes; ++p) {
        const uint32_t c = h[p][threadIdx.x];
        if (c) atomicAdd(&u.totals[p * kDigits + threadIdx.x], c);
    }
}

// Clears the statuses of the tiles of n keys (the grid shares them).
__device__ __forceinline__ void sort_status_clear(const SortUse& u, uint64_t n) {
    const uint64_t words = (n + u.tile - 1) / u.tile * kDigits;
    for (int p = 0; p < u.passes; ++p)
        for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < words;
             i += (uint64_t)gridDim.x * blockDim.x)
            u.status[p * u.status_pass + i] = 0;
}

}  // namespace btcx
