// Internal definitions shared by the host (.cpp) and device (.hip) sources of
// libbtc_amd.so.  Errors inside the library are raised as btcx::Error and
// turned into status codes at the C ABI (btcx::guard); nothing exits.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <new>
#include <vector>

#include "btc_amd.h"

namespace btcx {

struct Error {
    int code;
};

void set_error(const char* fmt, ...) __attribute__((format(printf, 1, 2)));
void clear_error();
[[noreturn]] void fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));

#define BTC_HIP(call)                                                                        \
    do {                                                                                     \
        hipError_t e_ = (call);                                                              \
        if (e_ != hipSuccess)                                                                \
            ::btcx::fail(e_ == hipErrorOutOfMemory ? BTC_ERR_NOMEM : BTC_ERR_HIP,            \
                         "%s: %s (%s:%d)", #call, hipGetErrorString(e_), __FILE__, __LINE__); \
    } while (0)

#define BTC_CHECK_LAUNCH(name)                                                                \
    do {                                                                                      \
        hipError_t e_ = hipGetLastError();                                                    \
        if (e_ != hipSuccess)                                                                 \
            ::btcx::fail(BTC_ERR_HIP, "launch of %s: %s", name, hipGetErrorString(e_));       \
    } while (0)

#define BTC_REQUIRE(cond, code, ...)          \
    do {                                      \
        if (!(cond)) ::btcx::fail(code, __VA_ARGS__); \
    } while (0)

// Rethrows a failed status of a nested C-ABI call (its message is kept).
inline void check_status(int rc) {
    if (rc != BTC_OK) throw Error{rc};
}

// Notes a call that failed, perhaps with work left on a stream (runtime.cpp).
void pool_call_failed();

// Runs f and maps library errors to status codes for the C ABI.
template <class F>
int guard(F&& f) {
    clear_error();
    try {
        f();
        return BTC_OK;
    } catch (const Error& e) {
        // bad arguments are refused before any work is enqueued, or on the
        // device's word once it has ended
        if (e.code != BTC_ERR_ARG) pool_call_failed();
        return e.code;
    } catch (const std::bad_alloc&) {
        pool_call_failed();
        set_error("host allocation failed");
        return BTC_ERR_NOMEM;
    } catch (...) {
        pool_call_failed();
        set_error("unexpected exception");
        return BTC_ERR_STATE;
    }
}

// Device memory behind DevBuf and TmpBuf: freed blocks are kept per device
// and handed out again (runtime.cpp has the rules), so the work of building
// a graph, a plan or a Bit-BSR is not spent in the allocator: hipFreeAsync
// waits for its stream and hipFree for the device, and together with the
// allocations they took 12 of the 21 ms of a build + count of an R-MAT 2^20
// graph and 2.0 of the 3.2 ms of a 64^3 stencil's from host pairs.
// `ordered`: the block's first (alloc) or last (free) use is in order on
// stream s; otherwise nothing is known about the stream, and the block is
// only reused once it is idle.  Neither call waits for the device (but for
// blocks that go back to the driver): a thread that builds a plan does not
// wait for the counts of others.
void* pool_alloc(size_t bytes, bool ordered, hipStream_t s);
void pool_free(void* p, bool ordered, hipStream_t s);

// Waits for the device, once, if blocks were released in no known order.
void pool_settle();

// Returns the current device's cached blocks to the driver; their bytes.
int64_t pool_release_all();

// hipStreamSynchronize at the end of a call: what the call released in order
// on s is idle then.
void stream_wait(hipStream_t s);

// Around the destruction of a handle: no entry point returns before its work
// has ended, so the handle's buffers are idle.  After a call that failed
// (pool_call_failed) they are taken to be in use until the device has been
// synchronised, which the scope's end does.
struct IdleScope {
    IdleScope();
    ~IdleScope();
    IdleScope(const IdleScope&) = delete;
    IdleScope& operator=(const IdleScope&) = delete;
};

template <class H>
void free_handle(H* h) {
    IdleScope scope;
    delete h;
}

// Owning device buffer (from the pool).
template <class T>
struct DevBuf {
    T* p = nullptr;
    size_t n = 0;
    bool owned = true;  // false: a view into memory that another buffer owns (view())
    DevBuf() = default;
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    DevBuf(DevBuf&& o) noexcept : p(o.p), n(o.n), owned(o.owned) { o.p = nullptr; o.n = 0; o.owned = true; }
    DevBuf& operator=(DevBuf&& o) noexcept {
        if (this != &o) {
            release();
            p = o.p;
            n = o.n;
            owned = o.owned;
            o.p = nullptr;
            o.n = 0;
            o.owned = true;
        }
        return *this;
    }
    // Points at count elements at q, which the buffer does not free.
    void view(T* q, size_t count) {
        release();
        p = q;
        n = count;
        owned = false;
    }
    ~DevBuf() { release(); }
    void alloc(size_t count) {
        release();
        if (count == 0) count = 1;  // keep a valid pointer for empty arrays
        p = static_cast<T*>(pool_alloc(count * sizeof(T), false, nullptr));
        n = count;
    }
    // alloc() for a buffer whose first use is in order on s
    void alloc_on(size_t count, hipStream_t s) {
        release();
        if (count == 0) count = 1;
        p = static_cast<T*>(pool_alloc(count * sizeof(T), true, s));
        n = count;
    }
    // release() of a buffer whose last use is in order on s
    void release_on(hipStream_t s) {
        if (p && owned) pool_free(p, true, s);
        p = nullptr;
        n = 0;
        owned = true;
    }
    void release() {
        if (p && owned) pool_free(p, false, nullptr);
        p = nullptr;
        n = 0;
        owned = true;
    }
    size_t bytes() const { return n * sizeof(T); }
};

// Keeps up to 1 GiB of freed stream-ordered memory cached in the current
// device's default pool (once per device), so temporaries are reused.
void mem_pool_init();

// A device arena for the temporary buffers (TmpBuf) of one thread's work on
// one stream: buffers are carved from one device block by a bump pointer
// (released in LIFO order, or all at once when the scope ends) and reused
// in stream order, so a thread that prepares many graphs (a server's
// preparation thread) makes no allocation call per buffer.  ArenaScope
// installs it for the calling thread and stream; buffers that do not fit
// come from the pool, and the block grows to the scope's demand (up
// to kArenaMax) when the scope ends.
struct Arena {
    char* base = nullptr;
    size_t cap = 0, top = 0, demand = 0;
    hipStream_t s = nullptr;
    Arena() = default;
    Arena(const Arena&) = delete;
    Arena& operator=(const Arena&) = delete;
    ~Arena();
};
constexpr size_t kArenaMax = size_t(1) << 30;

struct ArenaScope {
    Arena& a;
    Arena* prev;
    ArenaScope(Arena& arena, hipStream_t s);
    ~ArenaScope();
};

// The arena installed on this thread, or NULL.
Arena* current_arena();

// Stream-ordered temporary device buffer: from the thread's arena when one
// is installed for this stream, else from the pool, whose blocks a stream
// reuses in order (freeing waits for nothing, so threads that build plans
// side by side do not serialise on each other's kernels).
template <class T>
struct TmpBuf {
    T* p = nullptr;
    size_t n = 0;
    hipStream_t s = nullptr;
    size_t off = 0, bytes = 0;
    bool from_arena = false;
    TmpBuf() = default;
    TmpBuf(const TmpBuf&) = delete;
    TmpBuf& operator=(const TmpBuf&) = delete;
    ~TmpBuf() { release(); }
    void alloc(size_t count, hipStream_t stream) {
        release();
        if (count == 0) count = 1;
        s = stream;
        bytes = (count * sizeof(T) + 255) & ~size_t(255);
        Arena* a = current_arena();
        if (a && a->s == stream) {
            if (a->demand < a->top + bytes) a->demand = a->top + bytes;
            if (a->top + bytes <= a->cap) {
                off = a->top;
                p = reinterpret_cast<T*>(a->base + off);
                a->top += bytes;
                from_arena = true;
                n = count;
                return;
            }
        }
        p = static_cast<T*>(pool_alloc(count * sizeof(T), true, s));
        n = count;
    }
    // alloc() of an array that the caller can do without: false when there is
    // no memory for it
    bool try_alloc(size_t count, hipStream_t st) {
        try {
            alloc(count, st);
        } catch (const Error& e) {
            if (e.code != BTC_ERR_NOMEM) throw;
            clear_error();
            return false;
        }
        return true;
    }
    void release() {
        if (p) {
            if (!from_arena) {
                pool_free(p, true, s);
            } else {
                Arena* a = current_arena();
                if (a && off + bytes == a->top) a->top = off;  // the newest buffer: pop it
            }
        }
        p = nullptr;
        n = 0;
        from_arena = false;
    }
};

// Pinned host staging buffer, grown on demand (hipHostMalloc).
struct PinnedBuf {
    char* p = nullptr;
    size_t cap = 0;
    PinnedBuf() = default;
    PinnedBuf(const PinnedBuf&) = delete;
    PinnedBuf& operator=(const PinnedBuf&) = delete;
    ~PinnedBuf() {
        if (p) (void)hipHostFree(p);
    }
    char* reserve(size_t bytes);
};

// Pinned memory of the calling thread for what a call returns: the count
// kernels write a total (and a batch its graphs' sums) there themselves, so
// no copy to the host follows them.  host_words(bytes) may move the block
// when it grows: a call asks for its words before it takes host_total().
constexpr size_t kHostTotalBytes = 64;
char* host_words(size_t bytes);
unsigned long long* host_total();

// Copies count host arrays of `bytes` each into device memory (dev[k]) on
// stream s and waits: through a thread's cached pinned staging, two 16 MiB
// chunks at a time for large arrays (host threads fill one chunk while the
// DMA engine drains the other).
void upload_arrays(const void* const* host, void* const* dev, int count, size_t bytes, hipStream_t s);

// A HIP graph captured from a sequence of kernel launches, replayed with
// one hipGraphLaunch.  Captured work contains kernels only (buffers are
// cleared by fill kernels, not memset nodes).
struct CapturedGraph {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    CapturedGraph() = default;
    CapturedGraph(const CapturedGraph&) = delete;
    CapturedGraph& operator=(const CapturedGraph&) = delete;
    ~CapturedGraph() { reset(); }
    void reset() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        exec = nullptr;
        graph = nullptr;
    }
    // Captures what enqueue(stream) launches on a private stream.
    template <class F>
    void capture(F&& enqueue) {
        reset();
        hipStream_t cs = nullptr;
        BTC_HIP(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
        hipError_t e = hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal);
        if (e == hipSuccess) {
            try {
                enqueue(cs);
            } catch (...) {
                hipGraph_t g = nullptr;
                (void)hipStreamEndCapture(cs, &g);
                if (g) (void)hipGraphDestroy(g);
                (void)hipStreamDestroy(cs);
                throw;
            }
            e = hipStreamEndCapture(cs, &graph);
        }
        (void)hipStreamDestroy(cs);
        if (e == hipSuccess) e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        if (e != hipSuccess) {
            reset();
            (void)hipGetLastError();
            fail(BTC_ERR_HIP, "graph capture failed: %s", hipGetErrorString(e));
        }
    }
    void launch(hipStream_t s) { BTC_HIP(hipGraphLaunch(exec, s)); }
};

// Kernel timing with HIP events recorded on the launch stream.
struct EventTimer {
    hipEvent_t a = nullptr, b = nullptr;
    int dev = 0;
    bool on = false;
    explicit EventTimer(bool enable);
    ~EventTimer();
    void start(hipStream_t s);
    void stop(hipStream_t s);
    float ms();  // synchronises on the stop event
};

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

// Device address of the current device's static count workspace (looked up
// on the first call per device; btc_device_init makes that call).
unsigned long long* noalloc_workspace();

// Count totals of kernels with many workgroups: each workgroup adds its
// partial sum into one of kSlots u64 slots kSlotStride words (one 128-byte
// line) apart instead of into one address, where same-address atomics
// serialise in L2; launch_slot_sum then folds the slots into the total and
// clears them.  Every count clears its words (total, counters, slots) first.
constexpr int kSlots = 64;
constexpr int kSlotStride = 16;
constexpr size_t kSlotWords = (size_t)kSlots * kSlotStride;
// A count's device words: [0] total, [1] two u32 work-item counters, the
// slots from word kWorkSlots on.
constexpr size_t kWorkSlots = 16;
constexpr size_t kWorkWords = kWorkSlots + kSlotWords;

// Per-vertex sums on the device.  A vertex's count is at most C(d, 2) for
// its row length d, which fits int32 while d <= kPv32MaxRow; graphs with a
// longer row sum into 64-bit slots.  At most one pointer is set (none:
// totals only).  Every kernel adds a lane's or a group's partial sum with
// one atomic (pv_add).
constexpr int32_t kPv32MaxRow = 65536;

struct PvOut {
    int32_t* p32 = nullptr;
    unsigned long long* p64 = nullptr;
    __host__ __device__ bool on() const { return p32 != nullptr || p64 != nullptr; }
};

// A lane of the tile kernels sums its row's intersections with K / 4 tile
// columns in 32 bits; each is at most the longest row.
inline bool lane_sums_fit(int64_t max_row, int K) { return max_row * (K / 4) < (int64_t(1) << 32); }

// Device per-vertex sums for n vertices of a graph whose longest row is
// max_row (int32 slots when every count fits them, else 64-bit).
struct PvBuf {
    DevBuf<int32_t> b32;
    DevBuf<unsigned long long> b64;
    size_t n = 0;
    void alloc(size_t count, int32_t max_row) {
        n = count;
        if (max_row <= kPv32MaxRow) b32.alloc(count);
        else b64.alloc(count);
    }
    // for one count on s, which copy_out's wait ends (release_idle then)
    void alloc_on(size_t count, int32_t max_row, hipStream_t s) {
        n = count;
        if (max_row <= kPv32MaxRow) b32.alloc_on(count, s);
        else b64.alloc_on(count, s);
    }
    // after the wait for the work that used it (a failed call, whose stack
    // unwinds, leaves it to the destructors instead)
    void release_idle() {
        IdleScope scope;
        b32.release();
        b64.release();
    }
    PvOut out() const { return PvOut{b32.p, b64.p}; }
    bool wide() const { return b64.p != nullptr; }
    void* data() const { return b64.p ? (void*)b64.p : (void*)b32.p; }
    size_t bytes() const { return n * (b64.p ? 8 : 4); }
    // what copy_out takes of the thread's pinned words: everything up to
    // kStageMax, else nothing
    static constexpr size_t kStageMax = size_t(16) << 20;
    size_t staged() const { return bytes() <= kStageMax ? bytes() : 0; }
    // Copies the sums to host int32 (h32; BTC_ERR_OVERFLOW when a count
    // does not fit) or int64 (h64) after the work on s; synchronises s.
    void copy_out(int32_t* h32, int64_t* h64, hipStream_t s) const;
};

}  // namespace btcx

// Canonical lower-triangular graph L (CSR, ascending columns) on host and HBM.
struct btc_graph_s {
    int32_t n = 0;
    int32_t n_input = 0;
    int64_t m = 0;
    int32_t max_row = 0;
    uint32_t flags = 0;
    int64_t wedges = 0;
    int64_t merge_work = 0;
    bool on_host = true;           // rowptr / col / labels below are valid
    std::vector<int64_t> rowptr;   // n + 1
    std::vector<int32_t> col;      // m
    std::vector<int32_t> labels;   // canonical -> input id
    btcx::DevBuf<uint32_t> d_rowptr;  // n + 1 (m < 2^32 is enforced)
    btcx::DevBuf<int32_t> d_col;      // m + padding
    btcx::DevBuf<int32_t> d_labels;   // n, for graphs canonicalised on the device
    // one allocation behind the device arrays above (views into it) and,
    // for an exported pipeline run, behind its plan's arrays too
    btcx::DevBuf<unsigned char> block;
};

namespace btcx {
// Fills the derived statistics (rows, wedges, merge work) of g.
void graph_finalize(btc_graph_s* g);
// Canonicalises device-resident COO pairs into g (CSR and labels in HBM,
// statistics filled, host copies left empty until ensure_host).  With
// segs (ascending vertex offsets of up to 64 independent graphs, segs[0] =
// 0, back = n), each graph stays one contiguous vertex range, relabelled by
// degree within itself; csegs receives the ranges after compaction.
void canonicalise_device(const int32_t* src, const int32_t* dst, int64_t nnz, int32_t n, uint32_t flags,
                         hipStream_t s, btc_graph_s* g, const std::vector<int64_t>* segs,
                         std::vector<int64_t>* csegs);
// Makes the host CSR and labels of g valid (copies them from HBM once).
void ensure_host(btc_graph_s* g);
// Fills the auto fields of o from the autotuner's table when an entry
// matches g's features; returns whether one did.
bool tune_table_apply(const btc_graph_s* g, btc_count_opts* o);
}  // namespace btcx
