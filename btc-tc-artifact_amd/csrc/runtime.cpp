// Error state, version, device selection, event timing and the scalar
// dispatch rules shared by every path.
#include <omp.h>

#include <algorithm>
#include <atomic>
#include <cstdarg>
#include <chrono>
#include <cstring>
#include <deque>
#include <exception>
#include <list>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "common.h"

namespace btcx {

static thread_local char g_err[1024] = {0};

void set_error(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

void clear_error() { g_err[0] = 0; }

void fail(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    throw Error{code};
}

// Events of this thread that no timer holds, by device: creating and
// destroying a pair took 3 us of a small count.
struct TimerEvents {
    std::vector<hipEvent_t> free[64];
    ~TimerEvents() {
        for (auto& v : free)
            for (hipEvent_t e : v) (void)hipEventDestroy(e);
    }
};
static thread_local TimerEvents tl_events;

EventTimer::EventTimer(bool enable) : on(enable) {
    if (!on) return;
    BTC_HIP(hipGetDevice(&dev));
    auto take = [this] {
        hipEvent_t e = nullptr;
        if (dev < 64 && !tl_events.free[dev].empty()) {
            e = tl_events.free[dev].back();
            tl_events.free[dev].pop_back();
        } else {
            BTC_HIP(hipEventCreate(&e));
        }
        return e;
    };
    a = take();
    b = take();
}

EventTimer::~EventTimer() {
    for (hipEvent_t e : {a, b}) {
        if (!e) continue;
        if (dev < 64 && tl_events.free[dev].size() < 8) tl_events.free[dev].push_back(e);
        else (void)hipEventDestroy(e);
    }
}

void EventTimer::start(hipStream_t s) {
    if (on) BTC_HIP(hipEventRecord(a, s));
}

void EventTimer::stop(hipStream_t s) {
    if (on) BTC_HIP(hipEventRecord(b, s));
}

float EventTimer::ms() {
    if (!on) return 0.f;
    BTC_HIP(hipEventSynchronize(b));
    float t = 0.f;
    BTC_HIP(hipEventElapsedTime(&t, a, b));
    return t;
}

}  // namespace btcx

// ------------------------------------------------------------ device pool
namespace btcx {
namespace {

constexpr int kPoolDevices = 64;

// The queue of work that a use is in order on.  A handle names one, except
// hipStreamPerThread, which is a stream of its own in every host thread: a
// number per thread, never given twice, tells those apart.  (hipStreamLegacy
// and NULL are one stream under two handles: taken for two, which is safe.)
// A destroyed stream's handle may come back for a new stream; no work of the
// old one can be left on a block then, since every entry point waits for what
// it released in order before it returns, or releases it unordered.
struct Order {
    bool ordered = false;
    hipStream_t s = nullptr;
    uint64_t thread = 0;
    Order() = default;
    Order(bool in_order, hipStream_t stream) : ordered(in_order), s(stream) {
        static std::atomic<uint64_t> threads{0};
        static thread_local const uint64_t mine = ++threads;
        if (stream == hipStreamPerThread) thread = mine;
    }
    bool same(const Order& o) const { return ordered && o.ordered && s == o.s && thread == o.thread; }
};

// A freed block.  It may be handed out
//  * for work in the order its last use was in, or
//  * for any work when it is idle: released so (released == 0), or the device
//    or its stream has been synchronised after its release.
struct FreeBlock {
    void* p;
    size_t bytes;
    Order order;
    uint64_t released;  // position among the pool's releases, from 1
    std::chrono::steady_clock::time_point at;
};

// Bounded: at most kPoolKeep cached bytes per device (3 % of its memory) in at
// most kPoolBlocks blocks, the oldest going first; blocks that nothing took
// for kPoolIdle are returned by the calls that follow, up to kPoolIdleEach by
// each; and a failing allocation returns every cached block before it is
// tried once more.
constexpr size_t kPoolKeep = size_t(8) << 30;
constexpr size_t kPoolBlocks = 4096;
constexpr std::chrono::seconds kPoolIdle{10};
constexpr size_t kPoolIdleEach = 16;

struct Pool {
    std::mutex mu;
    using At = std::list<FreeBlock>::iterator;
    std::list<FreeBlock> cached;               // oldest release first
    std::map<size_t, std::deque<At>> by_size;  // the same blocks, each size's oldest first
    std::unordered_map<void*, size_t> live;    // bytes of every block handed out
    size_t cached_bytes = 0;
    uint64_t releases = 0, synced = 0;  // releases up to synced: device synchronised since
    uint64_t unordered = 0;             // the last release that was in no known order
    uint64_t failed_synced = 0;         // of g_failed: device synchronised since
    std::map<std::pair<hipStream_t, uint64_t>, uint64_t> stream_synced;  // as synced, by order

    bool idle(const FreeBlock& b) const {
        if (b.released <= synced) return true;
        if (!b.order.ordered) return false;
        const auto it = stream_synced.find({b.order.s, b.order.thread});
        return it != stream_synced.end() && b.released <= it->second;
    }
};

thread_local int tl_idle_scopes = 0;
std::atomic<uint64_t> g_failed{0};       // calls that failed, perhaps with work left on a stream
std::atomic<bool> g_unsettled{false};    // blocks may wait for pool_settle

// Never destroyed: buffers of static objects may outlive any order of
// destruction, and the driver takes the memory back with the process.
Pool* const g_pools = new Pool[kPoolDevices];

int pool_device() {
    int dev = 0;
    BTC_HIP(hipGetDevice(&dev));
    BTC_REQUIRE(dev >= 0 && dev < kPoolDevices, BTC_ERR_ARG, "device %d: memory is kept for devices 0-%d", dev,
                kPoolDevices - 1);
    return dev;
}

// Sizes are rounded up to eighths of a power of two (at least 512 bytes), up
// to 64 MiB, so that inputs of about one size share blocks; larger ones to
// 2 MiB.
size_t pool_round(size_t bytes) {
    if (bytes <= 512) return 512;
    if (bytes > (size_t(64) << 20)) return (bytes + (size_t(2) << 20) - 1) & ~((size_t(2) << 20) - 1);
    size_t p2 = 512;
    while (p2 * 2 < bytes) p2 *= 2;
    const size_t step = std::max<size_t>(p2 / 8, 256);
    return (bytes + step - 1) / step * step;
}

// Waits for the device.  In the relaxed capture mode, since the thread may
// not refuse the wait because of a capture elsewhere in the process.
bool device_wait() {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    const bool swapped = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
    const hipError_t e = hipDeviceSynchronize();
    if (swapped) (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (e != hipSuccess) (void)hipGetLastError();
    return e == hipSuccess;
}

// Takes the cached block for `want` bytes that wastes least (at most an eighth
// of them, or as much again up to 64 KiB), the newest of its size, or NULL.
void* pool_take(Pool& q, size_t want, const Order& order) {
    const size_t most = want <= (size_t(64) << 10) ? 2 * want : want + want / 8;
    for (auto sz = q.by_size.lower_bound(want); sz != q.by_size.end() && sz->first <= most; ++sz) {
        auto& same = sz->second;
        for (size_t k = same.size(); k-- > 0;) {
            const FreeBlock b = *same[k];
            if (!order.same(b.order) && !q.idle(b)) continue;
            q.live[b.p] = b.bytes;  // may throw: before the block leaves the cache
            q.cached.erase(same[k]);
            same.erase(same.begin() + (std::ptrdiff_t)k);
            if (same.empty()) q.by_size.erase(sz);
            q.cached_bytes -= b.bytes;
            return b.p;
        }
    }
    return nullptr;
}

void pool_keep(Pool& q, const FreeBlock& b) {
    auto& same = q.by_size[b.bytes];
    q.cached.push_back(b);
    try {
        same.push_back(std::prev(q.cached.end()));
    } catch (...) {
        q.cached.pop_back();
        throw;
    }
    q.cached_bytes += b.bytes;
}

// Blocks to give back now: the oldest beyond `keep` bytes or kPoolBlocks, and
// some of those idle for kPoolIdle.
std::vector<void*> pool_trim(Pool& q, size_t keep) {
    std::vector<void*> out;
    const auto now = std::chrono::steady_clock::now();
    while (!q.cached.empty()) {
        const FreeBlock& b = q.cached.front();
        const bool idle = now - b.at > kPoolIdle && out.size() < kPoolIdleEach;
        if (!idle && q.cached_bytes <= keep && q.cached.size() <= kPoolBlocks) break;
        out.push_back(b.p);
        q.cached_bytes -= b.bytes;
        const auto sz = q.by_size.find(b.bytes);
        sz->second.pop_front();  // the oldest of all is the oldest of its size
        if (sz->second.empty()) q.by_size.erase(sz);
        q.cached.pop_front();
    }
    return out;
}

void give_back(const std::vector<void*>& blocks) {
    for (void* p : blocks) (void)hipFree(p);  // waits for work that still uses it
}

}  // namespace

void* pool_alloc(size_t bytes, bool ordered, hipStream_t s) {
    const size_t want = pool_round(bytes);
    const Order order(ordered, s);
    Pool& q = g_pools[pool_device()];
    std::vector<void*> old;
    void* p = nullptr;
    {
        std::lock_guard<std::mutex> lk(q.mu);
        p = pool_take(q, want, order);
        old = pool_trim(q, kPoolKeep);
    }
    give_back(old);
    if (p) return p;
    hipError_t e = hipMalloc(&p, want);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        {
            std::lock_guard<std::mutex> lk(q.mu);
            old = pool_trim(q, 0);
        }
        give_back(old);
        e = hipMalloc(&p, bytes);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            fail(BTC_ERR_NOMEM, "hipMalloc of %zu bytes failed: %s", bytes, hipGetErrorString(e));
        }
        std::lock_guard<std::mutex> lk(q.mu);
        q.live[p] = bytes;
        return p;
    }
    std::lock_guard<std::mutex> lk(q.mu);
    q.live[p] = want;
    return p;
}

void pool_free(void* p, bool ordered, hipStream_t s) {
    if (!p) return;
    // a buffer of a call that failed half-way: work may be left on any stream
    const bool unwinding = std::uncaught_exceptions() > 0;
    if (unwinding) ordered = false;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) dev = 0;
    bool kept = false;
    try {  // called by destructors: no exception leaves
        std::vector<void*> old;
        for (int k = 0; k < kPoolDevices; ++k) {
            Pool& q = g_pools[(dev + k) % kPoolDevices];  // the current device's almost always
            std::lock_guard<std::mutex> lk(q.mu);
            const auto it = q.live.find(p);
            if (it == q.live.end()) continue;
            const size_t bytes = it->second;
            q.live.erase(it);
            if (bytes <= kPoolKeep / 4) {  // one block does not crowd out the rest
                // a handle's own buffer: idle, as no call leaves work behind it
                // (but for failed ones)
                const bool idle = !ordered && !unwinding && tl_idle_scopes > 0 && q.failed_synced == g_failed;
                const uint64_t at = idle ? 0 : ++q.releases;
                if (!ordered && !idle) {
                    q.unordered = at;
                    g_unsettled = true;
                }
                pool_keep(q, {p, bytes, Order(ordered, s), at, std::chrono::steady_clock::now()});
                kept = true;
                old = pool_trim(q, kPoolKeep);
            }
            break;
        }
        give_back(old);
    } catch (...) {
    }
    if (!kept) (void)hipFree(p);
}

IdleScope::IdleScope() { ++tl_idle_scopes; }

IdleScope::~IdleScope() {
    if (--tl_idle_scopes == 0) pool_settle();
}

void pool_settle() {
    if (!g_unsettled) return;  // no HIP call: handles that never saw a device are freed too
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kPoolDevices) return;
    Pool& q = g_pools[dev];
    uint64_t upto, failed;
    {
        std::lock_guard<std::mutex> lk(q.mu);
        if (q.unordered <= q.synced) return;  // another device's
        upto = q.releases;
        failed = g_failed;
        g_unsettled = false;
    }
    const bool ok = device_wait();
    std::lock_guard<std::mutex> lk(q.mu);
    if (ok) {
        q.synced = std::max(q.synced, upto);
        q.failed_synced = std::max(q.failed_synced, failed);
    } else {
        g_unsettled = true;
    }
}

void pool_call_failed() { ++g_failed; }

int64_t pool_release_all() {
    Pool& q = g_pools[pool_device()];
    std::vector<void*> all;
    size_t bytes;
    {
        std::lock_guard<std::mutex> lk(q.mu);
        bytes = q.cached_bytes;
        all = pool_trim(q, 0);
    }
    give_back(all);
    return (int64_t)bytes;
}

void stream_wait(hipStream_t s) {
    Pool& q = g_pools[pool_device()];
    uint64_t upto;  // before the wait: other threads may use the stream meanwhile
    {
        std::lock_guard<std::mutex> lk(q.mu);
        upto = q.releases;
    }
    BTC_HIP(hipStreamSynchronize(s));
    const Order o(true, s);
    std::lock_guard<std::mutex> lk(q.mu);
    if (q.stream_synced.size() >= 1024) q.stream_synced.clear();  // handles and threads come and go
    uint64_t& at = q.stream_synced[{o.s, o.thread}];
    at = std::max(at, upto);
}

void mem_pool_init() {
    static std::once_flag once[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return;
    std::call_once(once[dev], [dev] {
        hipMemPool_t pool = nullptr;
        if (hipDeviceGetDefaultMemPool(&pool, dev) != hipSuccess) {
            (void)hipGetLastError();
            return;
        }
        uint64_t keep = 1ull << 30;
        (void)hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep);
        (void)hipGetLastError();
    });
}

static thread_local Arena* tl_arena = nullptr;

Arena* current_arena() { return tl_arena; }

Arena::~Arena() {
    if (base) (void)hipFreeAsync(base, s);
}

ArenaScope::ArenaScope(Arena& arena, hipStream_t s) : a(arena), prev(tl_arena) {
    a.s = s;
    a.top = 0;
    a.demand = 0;
    tl_arena = &a;
}

ArenaScope::~ArenaScope() {
    tl_arena = prev;
    a.top = 0;
    if (a.demand > a.cap && a.cap < kArenaMax) {
        // grow to the scope's demand (a power of two, at least 64 MiB)
        size_t c = size_t(64) << 20;
        while (c < a.demand && c < kArenaMax) c <<= 1;
        if (a.base) (void)hipFreeAsync(a.base, a.s);
        a.base = nullptr;
        a.cap = 0;
        mem_pool_init();
        if (hipMallocAsync(reinterpret_cast<void**>(&a.base), c, a.s) == hipSuccess) a.cap = c;
        else (void)hipGetLastError();  // the arena stays empty: buffers come from the pool
    }
}

char* PinnedBuf::reserve(size_t bytes) {
    if (bytes <= cap) return p;
    size_t c = size_t(1) << 20;
    while (c < bytes) c <<= 1;
    if (p) (void)hipHostFree(p);
    p = nullptr;
    cap = 0;
    BTC_HIP(hipHostMalloc(reinterpret_cast<void**>(&p), c, hipHostMallocDefault));
    cap = c;
    return p;
}

void upload_arrays(const void* const* host, void* const* dev, int count, size_t bytes, hipStream_t s) {
    constexpr size_t kChunk = size_t(16) << 20;
    if (bytes == 0) return;
    if (bytes <= kChunk / 4) {  // small: one staging copy each
        static thread_local PinnedBuf small;
        char* b = small.reserve(bytes * (size_t)count);
        for (int k = 0; k < count; ++k) {
            std::memcpy(b + (size_t)k * bytes, host[k], bytes);
            BTC_HIP(hipMemcpyAsync(dev[k], b + (size_t)k * bytes, bytes, hipMemcpyHostToDevice, s));
        }
        BTC_HIP(hipStreamSynchronize(s));
        return;
    }
    // two pinned chunks: host threads fill one while the DMA engine drains
    // the other (each chunk's event says when it may be refilled)
    static thread_local PinnedBuf stage;
    char* buf = stage.reserve(2 * kChunk);
    hipEvent_t done[2] = {nullptr, nullptr};
    BTC_HIP(hipEventCreateWithFlags(&done[0], hipEventDisableTiming));
    hipError_t e = hipEventCreateWithFlags(&done[1], hipEventDisableTiming);
    if (e != hipSuccess) {
        (void)hipEventDestroy(done[0]);
        BTC_HIP(e);
    }
    bool used[2] = {false, false};
    int slot = 0;
    e = hipSuccess;
    for (int k = 0; k < count && e == hipSuccess; ++k) {
        const char* src = static_cast<const char*>(host[k]);
        char* dst = static_cast<char*>(dev[k]);
        for (size_t off = 0; off < bytes && e == hipSuccess; off += kChunk) {
            const size_t len = std::min(kChunk, bytes - off);
            char* c = buf + (size_t)slot * kChunk;
            if (used[slot]) e = hipEventSynchronize(done[slot]);
            if (e != hipSuccess) break;
            const int parts = (int)std::max<size_t>(1, std::min<size_t>(16, len >> 20));
#pragma omp parallel for num_threads(parts) schedule(static)
            for (int t = 0; t < parts; ++t) {
                const size_t a = len * (size_t)t / (size_t)parts, b = len * (size_t)(t + 1) / (size_t)parts;
                std::memcpy(c + a, src + off + a, b - a);
            }
            e = hipMemcpyAsync(dst + off, c, len, hipMemcpyHostToDevice, s);
            if (e == hipSuccess) e = hipEventRecord(done[slot], s);
            used[slot] = true;
            slot ^= 1;
        }
    }
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    (void)hipEventDestroy(done[0]);
    (void)hipEventDestroy(done[1]);
    BTC_HIP(e);
}

// 64-bit sums to int32, each checked.
static void narrow_sums(const unsigned long long* t, size_t n, int32_t* h32) {
    for (size_t v = 0; v < n; ++v) {
        BTC_REQUIRE(t[v] <= (unsigned long long)INT32_MAX, BTC_ERR_OVERFLOW,
                    "vertex %zu closes %llu triangles, beyond int32 per-vertex output (the int64 entry points "
                    "return it)", v, t[v]);
        h32[v] = (int32_t)t[v];
    }
}

char* host_words(size_t bytes) {
    static thread_local PinnedBuf words;
    return words.reserve(bytes + kHostTotalBytes) + kHostTotalBytes;
}

unsigned long long* host_total() { return reinterpret_cast<unsigned long long*>(host_words(0) - kHostTotalBytes); }

void PvBuf::copy_out(int32_t* h32, int64_t* h64, hipStream_t s) const {
    if (n == 0 || (!h32 && !h64)) {
        BTC_HIP(hipStreamSynchronize(s));
        return;
    }
    // up to kStageMax bytes come through pinned memory of the thread (a copy
    // to pageable memory is staged by the runtime at a third of the rate)
    if (staged()) {
        const void* d = b64.p ? (const void*)b64.p : (const void*)b32.p;
        char* const pin = host_words(bytes());
        BTC_HIP(hipMemcpyAsync(pin, d, bytes(), hipMemcpyDeviceToHost, s));
        BTC_HIP(hipStreamSynchronize(s));
        if (wide() == (h64 != nullptr)) {
            char* const out = h64 ? reinterpret_cast<char*>(h64) : reinterpret_cast<char*>(h32);
            const size_t total = bytes(), parts = std::min<size_t>((size_t)omp_get_max_threads(), std::max<size_t>(1, std::min<size_t>(8, total >> 17)));
#pragma omp parallel for num_threads((int)parts) if (parts > 1) schedule(static)
            for (size_t t = 0; t < parts; ++t) {
                const size_t a = total * t / parts, z = total * (t + 1) / parts;
                std::memcpy(out + a, pin + a, z - a);
            }
        } else if (h64) {
            const int32_t* t = reinterpret_cast<const int32_t*>(pin);
            for (size_t v = 0; v < n; ++v) h64[v] = t[v];
        } else {
            narrow_sums(reinterpret_cast<const unsigned long long*>(pin), n, h32);
        }
        return;
    }
    if (!wide() && h32) {
        BTC_HIP(hipMemcpyAsync(h32, b32.p, n * 4, hipMemcpyDeviceToHost, s));
        BTC_HIP(hipStreamSynchronize(s));
        return;
    }
    if (wide() && h64) {
        BTC_HIP(hipMemcpyAsync(h64, b64.p, n * 8, hipMemcpyDeviceToHost, s));
        BTC_HIP(hipStreamSynchronize(s));
        return;
    }
    if (h64) {  // int32 slots widened
        std::vector<int32_t> t(n);
        BTC_HIP(hipMemcpyAsync(t.data(), b32.p, n * 4, hipMemcpyDeviceToHost, s));
        BTC_HIP(hipStreamSynchronize(s));
        for (size_t v = 0; v < n; ++v) h64[v] = t[v];
        return;
    }
    std::vector<unsigned long long> t(n);  // 64-bit slots narrowed, each checked
    BTC_HIP(hipMemcpyAsync(t.data(), b64.p, n * 8, hipMemcpyDeviceToHost, s));
    BTC_HIP(hipStreamSynchronize(s));
    narrow_sums(t.data(), n, h32);
}

}  // namespace btcx

extern "C" {

const char* btc_last_error(void) { return btcx::g_err; }

const char* btc_version(void) { return "0.1.0-gfx950"; }

int btc_memory_trim(int64_t* released_bytes) {
    return btcx::guard([&] {
        const int64_t bytes = btcx::pool_release_all();
        if (released_bytes) *released_bytes = bytes;
    });
}

int btc_device_init(int32_t device) {
    return btcx::guard([&] {
        int count = 0;
        hipError_t e = hipGetDeviceCount(&count);
        if (e != hipSuccess || count == 0) {
            (void)hipGetLastError();
            btcx::fail(BTC_ERR_HIP, "no HIP device available");
        }
        BTC_REQUIRE(device >= 0 && device < count, BTC_ERR_ARG, "device %d out of range [0,%d)",
                    device, count);
        BTC_HIP(hipSetDevice(device));
        btcx::noalloc_workspace();  // once per device, with the device current
    });
}

// apps/btc_tc_lite.cu:45-65: 16x32 if the average L-row is below 15 or the
// graph has fewer than 50,000 rows, else 16x128; BTC_MODE 1/2 force 32/128.
int32_t btc_lite_tile_k(int32_t n, int64_t m, int32_t mode) {
    if (mode == 1) return 32;
    if (mode == 2) return 128;
    if (n <= 0) return 32;
    float avg = (float)m / (float)n;
    return (avg < 15.0f || n < 50000) ? 32 : 128;
}

// tau literals: tc_16x128_mma_v5.h:51 (512 of 2048 bits), tc_16x32_mma_v6.h:52
// (64 of 512 bits); 16x64 is not in the reference and takes 12.5 % (128 of 1024).
int32_t btc_default_tau(int32_t tile_k) {
    switch (tile_k) {
        case 128: return 512;
        case 64: return 128;
        case 32: return 64;
        default: return -1;
    }
}

}  // extern "C"
