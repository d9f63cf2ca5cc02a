// Device-wide sort and scan used by the device canonicaliser and planner
// (rocPRIM underneath; kept in one translation unit for compile time).
// Every function runs on `s` and returns once the work is enqueued; its
// temporary storage is allocated and freed in stream order on `s`.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace btcx {

// Sorts keys[0, n) ascending on bits [0, end_bit); tmp holds n keys.
// Returns the buffer that holds the result (keys or tmp).
uint64_t* sort_u64(uint64_t* keys, uint64_t* tmp, size_t n, int end_bit, hipStream_t s);

// Stable sort of (key, value) pairs on key bits [0, end_bit); kt / vt hold n
// entries each.  Returns whether the result is in (kt, vt) rather than
// (keys, vals).
bool sort_pairs_u32(uint32_t* keys, uint32_t* vals, uint32_t* kt, uint32_t* vt, size_t n, int end_bit,
                    hipStream_t s);

// out[i] = sum of in[0, i) for i <= n (out has n + 1 entries; out[n] = total).
void exclusive_scan_u32(const uint32_t* in, uint32_t* out, size_t n, hipStream_t s);
void exclusive_scan_u64(const uint64_t* in, uint64_t* out, size_t n, hipStream_t s);

// Capturable forms (devprim.hip, devtile.h).  The element count n is read
// from device memory (*d_n) when the kernels run, buffers hold `cap` elements
// (n <= cap), and a workspace (dseq_bytes(cap) bytes, 256-byte aligned)
// holds every temporary: kernels are the only work enqueued, so one stream
// capture serves every n up to cap.
//
// A run of sorts and scans in stream order takes its uses from one DevSeq
// when it is enqueued: each has tickets, totals and scan statuses of its
// own, all of them in the words [0, dseq_clear_words) that the run's first
// kernel clears (but for word kSeqErr, which stays).  A sort's statuses are
// shared by all and cleared by the kernel that writes its keys.
// Keys of a sort's tile, by capacity: large inputs pay for tickets and
// look-back per tile, small ones for CUs without a tile (replays of one graph
// of 131 K / 524 K / 1.6 M pairs with tiles of 2048 against 4096: 258 / 408 /
// 964 us against 282 / 413 / 880, a group of 3.3 M 1914 against 1678).
constexpr uint32_t kSortTileMin = 2048, kSortTileMax = 4096;
inline uint32_t sort_tile(size_t cap) { return cap > (size_t(1) << 20) ? kSortTileMax : kSortTileMin; }
constexpr int kMaxSorts = 6, kMaxScans = 8;
constexpr uint32_t kSeqErr = 0;
struct SortUse;
struct ScanUse;
struct DevSeq {
    void* p = nullptr;
    size_t cap = 0;
    int sorts = 0, scans = 0;
};
size_t dseq_bytes(size_t cap);
size_t dseq_clear_words(size_t cap);
SortUse dseq_sort(DevSeq& q, int end_bit);
ScanUse dseq_scan(DevSeq& q);

// Word that a sort or scan sets (and nothing clears) if a look-back ever ran
// past its spin limit -- a result that cannot be trusted.
const uint32_t* dseq_error_word(const DevSeq& q);

// The passes of a stable radix sort whose keys' writer filled in u.  u64
// keys: returns the buffer that holds the result; pairs: whether the result
// is in (kt, vt).
uint64_t* dsort_u64(uint64_t* keys, uint64_t* tmp, size_t cap, const uint32_t* d_n, const SortUse& u, hipStream_t s);
bool dsort_pairs_u32(uint32_t* keys, uint32_t* vals, uint32_t* kt, uint32_t* vt, size_t cap, const uint32_t* d_n,
                     const SortUse& u, hipStream_t s);

}  // namespace btcx
