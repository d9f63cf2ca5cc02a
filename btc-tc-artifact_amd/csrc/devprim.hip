// Radix sort whose key count is read from device memory when the kernels
// run.  It enqueues kernels only -- no allocation, no memset node, no host
// synchronisation -- so a stream capture of it replays for any count up to
// the capacity its buffers were sized for (see prim.h).
//
// Least-significant-digit, 8 bits a pass, in one sweep per pass: the kernel
// that writes the keys takes the digit totals of every pass on the way
// (devtile.h); each pass kernel then ranks a tile stably in LDS (rocPRIM's
// block_radix_rank, match form: per-wave ballots of equal digits) and finds
// the tile's offset for each digit by decoupled look-back.  A pass of 131 K
// u64 keys takes 10 us and one of 3.3 M 41 us (11 and 75 with two tickets a
// workgroup, a finish counter and a histogram kernel's own read of the keys):
// tickets and look-back round trips, not the 53 MB moved, bound the latter.
#include <rocprim/block/block_radix_rank.hpp>

#include "common.h"
#include "devtile.h"

namespace btcx {
namespace {

constexpr int kT = kTileThreads;

size_t tiles(size_t cap, size_t tile) { return std::max<size_t>(1, (cap + tile - 1) / tile); }

// Exclusive scan of one value per thread of a 256-thread workgroup.
__device__ uint32_t block_scan_ex(uint32_t v, uint32_t* lds) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) lds[wid] = x;
    __syncthreads();
    uint32_t base = 0;
#pragma unroll
    for (int w = 0; w < kT / 64; ++w)
        if (w < wid) base += lds[w];
    __syncthreads();
    return base + x - v;
}

// Workspace layout (256-byte aligned parts): control words (the error word,
// then each use's tickets), each sort's digit totals, each scan's tile
// statuses, then the statuses all sorts share.
constexpr uint32_t kSortTickets = 64;                                // + kMaxPasses per sort
constexpr uint32_t kScanTickets = kSortTickets + 16 * kMaxSorts;     // + 16 per scan, 64 bytes apart
constexpr uint32_t kCtlWords = (kScanTickets + 16 * kMaxScans + 63) / 64 * 64;
constexpr size_t kTotalsWords = (size_t)kMaxPasses * kDigits;
static_assert(kMaxPasses <= 16, "tickets of a sort");

size_t scan_words(size_t cap) { return (2 * tiles(cap, 2 * kTileThreads) + 63) & ~size_t(63); }  // smallest tiles

// Sum of the values of tiles [0, t) for one digit, by one thread: kLookAhead
// tiles' cells are read together.
constexpr int kLookAhead = 4;
__device__ __forceinline__ uint64_t look_back(const uint64_t* cells, int64_t j0, size_t stride, uint32_t* err) {
    uint64_t excl = 0;
    for (int64_t j = j0; j >= 0; j -= kLookAhead) {
        uint64_t x[kLookAhead];
#pragma unroll
        for (int k = 0; k < kLookAhead; ++k) x[k] = j >= k ? tile_load(cells + (size_t)(j - k) * stride) : kTileInc;
        bool done = false;
#pragma unroll
        for (int k = 0; k < kLookAhead; ++k) {
            if (done) continue;
            if ((x[k] >> 62) == 0) x[k] = tile_settle(cells + (size_t)(j - k) * stride, x[k], err);
            excl += x[k] & kTileMask;
            done = (x[k] >> 62) == 2;
        }
        if (done) break;
    }
    return excl;
}

// One stable pass.  Workgroups take tiles in ticket order; a tile ranks its
// keys in LDS (rocPRIM's block_radix_rank, match form), publishes its count
// of each digit and looks back over earlier tiles for the digit's offset
// (thread d owns digit d), then writes its keys out run by run.  Key i of a
// tile sits at index wave * 64 * kSortPer + item * 64 + lane, the order in
// which the match ranking breaks ties, so equal digits keep their input
// order; padding keys (all bits set) rank after every real key of the tile.
// Every look-back ends: a ticket is only taken by a running workgroup,
// which publishes before it waits on anything.
template <class K, bool V, int kSortPer>
__global__ __launch_bounds__(kT) void dsort_onesweep(const K* __restrict__ kin, const uint32_t* __restrict__ vin,
                                                     K* __restrict__ kout, uint32_t* __restrict__ vout,
                                                     const uint32_t* __restrict__ d_n, int pass, SortUse u) {
    constexpr uint32_t kSortTile = kT * kSortPer;
    using Rank = rocprim::block_radix_rank<kT, kDigitBits, rocprim::block_radix_rank_algorithm::match>;
    static_assert(Rank::digits_per_thread == 1, "one digit per thread");
    __shared__ typename Rank::storage_type rank_lds;
    __shared__ K sk[kSortTile];
    __shared__ uint32_t sv[V ? kSortTile : 1];
    __shared__ uint32_t s_pre[kDigits], s_out[kDigits];
    __shared__ uint32_t s_scan[kT / 64];
    __shared__ uint32_t s_tile;
    const int shift = pass * kDigitBits;
    const uint32_t n = *d_n, nt = (n + kSortTile - 1) / kSortTile;
    if (blockIdx.x >= nt) return;  // workgroup-uniform
    const uint32_t lane = threadIdx.x & 63, wid = threadIdx.x >> 6, d = threadIdx.x;
    const uint32_t dstart = block_scan_ex(u.totals[pass * kDigits + d], s_scan);
    uint64_t* const status = u.status + (size_t)pass * u.status_pass;
    for (TileLoop l(u.tickets + pass, nt, &s_tile); l.next();) {
        const uint32_t t = l.t;
        const size_t base = (size_t)t * kSortTile;
        const uint32_t valid = (uint32_t)min((size_t)kSortTile, (size_t)n - base);
        K k[kSortPer];
        uint32_t v[kSortPer], r[kSortPer];
#pragma unroll
        for (int i = 0; i < kSortPer; ++i) {
            const uint32_t idx = wid * (64 * kSortPer) + i * 64 + lane;
            k[i] = idx < valid ? kin[base + idx] : ~K(0);
            if constexpr (V) v[i] = idx < valid ? vin[base + idx] : 0u;
        }
        uint32_t pre[1], cnt[1];
        Rank().rank_keys(k, r, rank_lds, [shift](const K& x) { return digit_of(x, shift); }, pre, cnt);
        uint64_t* mine = status + (size_t)t * kDigits + d;
        uint32_t excl = 0;
        if (t == 0) {
            tile_store(mine, kTileInc | cnt[0]);
        } else {
            tile_store(mine, kTileAgg | cnt[0]);
            excl = (uint32_t)look_back(status + d, (int64_t)t - 1, kDigits, u.err);
            tile_store(mine, kTileInc | (uint64_t)(excl + cnt[0]));
        }
#pragma unroll
        for (int i = 0; i < kSortPer; ++i) {
            sk[r[i]] = k[i];
            if constexpr (V) sv[r[i]] = v[i];
        }
        s_pre[d] = pre[0];
        s_out[d] = dstart + excl;
        __syncthreads();
        for (uint32_t idx = threadIdx.x; idx < valid; idx += kT) {
            const K x = sk[idx];
            const uint32_t dx = digit_of(x, shift);
            const uint32_t pos = s_out[dx] + idx - s_pre[dx];
            if (pos >= n) continue;  // unreachable when the counts agree; keeps a bad count in bounds
            kout[pos] = x;
            if constexpr (V) vout[pos] = sv[idx];
        }
    }
}

// Returns whether the result is in (kt, vt).
template <class K, bool V>
bool dsort_t(K* keys, uint32_t* vals, K* kt, uint32_t* vt, size_t cap, const uint32_t* d_n, const SortUse& u,
             hipStream_t s) {
    const unsigned g = (unsigned)std::min<size_t>(tiles(cap, u.tile), 2048);  // tiles go by ticket
    K* ki = keys;
    K* ko = kt;
    uint32_t* vi = vals;
    uint32_t* vo = vt;
    for (int p = 0; p < u.passes; ++p) {
        if (u.tile == kSortTileMin)
            hipLaunchKernelGGL((dsort_onesweep<K, V, kSortTileMin / kT>), dim3(g), dim3(kT), 0, s, ki, vi, ko, vo, d_n, p, u);
        else
            hipLaunchKernelGGL((dsort_onesweep<K, V, kSortTileMax / kT>), dim3(g), dim3(kT), 0, s, ki, vi, ko, vo, d_n, p, u);
        BTC_CHECK_LAUNCH("dsort_onesweep");
        std::swap(ki, ko);
        std::swap(vi, vo);
    }
    return u.passes & 1;
}

}  // namespace

size_t dseq_clear_words(size_t cap) { return kCtlWords + kMaxSorts * kTotalsWords + kMaxScans * scan_words(cap); }

size_t dseq_bytes(size_t cap) {
    return dseq_clear_words(cap) * 4 + (size_t)kMaxPasses * tiles(cap, sort_tile(cap)) * kDigits * 8;
}

SortUse dseq_sort(DevSeq& q, int end_bit) {
    BTC_REQUIRE(q.sorts < kMaxSorts, BTC_ERR_STATE, "more than %d sorts in a run", kMaxSorts);
    const int passes = (std::max(end_bit, 0) + kDigitBits - 1) / kDigitBits;
    BTC_REQUIRE(passes <= kMaxPasses, BTC_ERR_ARG, "sort on %d bits", end_bit);
    auto* w = static_cast<uint32_t*>(q.p);
    const int k = q.sorts++;
    return SortUse{w + kSortTickets + 16 * k,
                   w + kCtlWords + (size_t)k * kTotalsWords,
                   reinterpret_cast<uint64_t*>(w + dseq_clear_words(q.cap)),
                   tiles(q.cap, sort_tile(q.cap)) * kDigits,
                   w + kSeqErr,
                   passes,
                   sort_tile(q.cap)};
}

ScanUse dseq_scan(DevSeq& q) {
    BTC_REQUIRE(q.scans < kMaxScans, BTC_ERR_STATE, "more than %d scans in a run", kMaxScans);
    auto* w = static_cast<uint32_t*>(q.p);
    const int k = q.scans++;
    return ScanUse{w + kScanTickets + 16 * k,
                   reinterpret_cast<uint64_t*>(w + kCtlWords + kMaxSorts * kTotalsWords +
                                               (size_t)k * scan_words(q.cap)),
                   w + kSeqErr};
}

const uint32_t* dseq_error_word(const DevSeq& q) { return static_cast<const uint32_t*>(q.p) + kSeqErr; }

uint64_t* dsort_u64(uint64_t* keys, uint64_t* tmp, size_t cap, const uint32_t* d_n, const SortUse& u, hipStream_t s) {
    return dsort_t<uint64_t, false>(keys, nullptr, tmp, nullptr, cap, d_n, u, s) ? tmp : keys;
}

bool dsort_pairs_u32(uint32_t* keys, uint32_t* vals, uint32_t* kt, uint32_t* vt, size_t cap, const uint32_t* d_n,
                     const SortUse& u, hipStream_t s) {
    return dsort_t<uint32_t, true>(keys, vals, kt, vt, cap, d_n, u, s);
}

}  // namespace btcx
