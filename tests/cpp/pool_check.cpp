// The device memory pool of csrc/runtime.cpp over a host stand-in for the HIP
// calls it makes: "device" blocks are numbered addresses that nothing
// dereferences, and every call is counted.  Each check is a run of its own
// (argv[1]), so that it starts with an empty pool.  Prints "pool ok".
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <memory>
#include <set>
#include <string>
#include <thread>
#include <vector>

#include "common.h"

// ------------------------------------------------------------- stand-in
namespace {
std::atomic<int> mallocs{0}, frees{0}, waits{0};
size_t in_use = 0, capacity = size_t(1) << 50;
uintptr_t next_address = uintptr_t(1) << 40;
std::vector<std::pair<uintptr_t, size_t>> blocks;
std::function<void()> during_sync;
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) {
    ++mallocs;
    if (in_use + bytes > capacity) return hipErrorOutOfMemory;
    in_use += bytes;
    *p = reinterpret_cast<void*>(next_address);
    blocks.emplace_back(next_address, bytes);
    next_address += (bytes + 4095) / 4096 * 4096;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    ++frees;
    for (auto& b : blocks)
        if (b.first == reinterpret_cast<uintptr_t>(p)) {
            in_use -= b.second;
            b = blocks.back();
            blocks.pop_back();
            return hipSuccess;
        }
    std::fprintf(stderr, "hipFree of %p, which is not allocated\n", p);
    std::abort();
}
hipError_t hipDeviceSynchronize() {
    ++waits;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    if (during_sync) during_sync();
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
// not reached by the checks
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t*, int) { return hipErrorNotSupported; }
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void*) { return hipErrorNotSupported; }
hipError_t hipMallocAsync(void**, size_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipFreeAsync(void*, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipEventCreate(hipEvent_t*) { return hipErrorNotSupported; }
hipError_t hipEventCreateWithFlags(hipEvent_t*, unsigned) { return hipErrorNotSupported; }
hipError_t hipEventDestroy(hipEvent_t) { return hipErrorNotSupported; }
hipError_t hipEventElapsedTime(float*, hipEvent_t, hipEvent_t) { return hipErrorNotSupported; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipErrorNotSupported; }
hipError_t hipHostFree(void*) { return hipErrorNotSupported; }
hipError_t hipHostMalloc(void**, size_t, unsigned) { return hipErrorNotSupported; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipErrorNotSupported; }
}

namespace btcx {
unsigned long long* noalloc_workspace() { std::abort(); }
}  // namespace btcx

namespace {

int failures = 0;

#define EXPECT(cond)                                                                          \
    do {                                                                                      \
        if (!(cond)) {                                                                        \
            std::fprintf(stderr, "%s:%d: check failed: %s\n", __FILE__, __LINE__, #cond);     \
            ++failures;                                                                       \
        }                                                                                     \
    } while (0)

hipStream_t stream(int k) { return reinterpret_cast<hipStream_t>(uintptr_t(0x1000) + 64 * (uintptr_t)k); }

void on_thread(const std::function<void()>& f) {
    std::thread t(f);
    t.join();
}

using btcx::pool_alloc;
using btcx::pool_free;

// One handle value, another stream in each thread: a block that one thread
// released in order is not handed to another without a wait for the device,
// nor to a later thread that the system gave the first one's identity.
void per_thread_stream() {
    void* a = pool_alloc(4096, true, hipStreamPerThread);
    pool_free(a, true, hipStreamPerThread);
    on_thread([&] {
        const int before = waits;
        void* b = pool_alloc(4096, true, hipStreamPerThread);
        EXPECT(b != a || waits > before);
        pool_free(b, true, hipStreamPerThread);
        void* c = pool_alloc(4096, true, hipStreamPerThread);
        EXPECT(c == b);  // its own stream's order
        pool_free(c, true, hipStreamPerThread);
    });
    for (int k = 0; k < 8; ++k) {
        void* last = nullptr;
        on_thread([&] {
            last = pool_alloc(65536, true, hipStreamPerThread);
            pool_free(last, true, hipStreamPerThread);
        });
        on_thread([&] {
            const int before = waits;
            void* b = pool_alloc(65536, true, hipStreamPerThread);
            EXPECT(b != last || waits > before);
            pool_free(b, true, hipStreamPerThread);
        });
    }
    // one stream shared by threads stays one order
    void* x = pool_alloc(1 << 20, true, stream(1));
    pool_free(x, true, stream(1));
    on_thread([&] {
        const int before = waits;
        void* y = pool_alloc(1 << 20, true, stream(1));
        EXPECT(y == x && waits == before);
        pool_free(y, true, stream(1));
    });
}

// An allocation never waits for the device: blocks that work of another
// stream, or of no known one, may still use are left alone.  pool_settle waits
// once for all of them.
void no_waits() {
    void* a = pool_alloc(1 << 16, true, stream(1));
    pool_free(a, true, stream(1));
    void* b = pool_alloc(1 << 16, true, stream(2));
    EXPECT(b != a && waits == 0);
    btcx::pool_settle();  // nothing was released in no known order
    EXPECT(waits == 0);
    pool_free(b, false, nullptr);
    void* c = pool_alloc(1 << 16, false, nullptr);
    void* d = pool_alloc(1 << 16, true, stream(2));
    EXPECT(c != a && c != b && d != a && d != b && waits == 0);
    btcx::pool_settle();
    EXPECT(waits == 1);
    btcx::pool_settle();
    EXPECT(waits == 1);
    const std::set<void*> idle{a, b};
    void* e = pool_alloc(1 << 16, false, nullptr);
    void* f = pool_alloc(1 << 16, true, stream(3));
    EXPECT(idle.count(e) && idle.count(f) && e != f && waits == 1);
    for (void* p : {c, d, e, f}) pool_free(p, false, nullptr);
    btcx::pool_settle();
    EXPECT(waits == 2 && mallocs == 4);
}

struct Handle {
    btcx::DevBuf<char> x;
};

Handle* make(hipStream_t s) {
    auto* h = new Handle;
    h->x.alloc_on(1 << 16, s);
    return h;
}

// A handle's buffers are idle when it is freed: no wait, and any stream may
// have them next.  After a call that failed with work enqueued, perhaps, the
// free waits, and the next one need not; bad arguments are not such a call.
void handles() {
    Handle* h = make(stream(1));
    void* a = h->x.p;
    btcx::free_handle(h);
    EXPECT(waits == 0);
    h = make(stream(2));
    EXPECT(h->x.p == a && waits == 0);
    EXPECT(btcx::guard([] { btcx::fail(BTC_ERR_ARG, "refused"); }) == BTC_ERR_ARG);
    btcx::free_handle(h);
    EXPECT(waits == 0);
    h = make(stream(3));
    EXPECT(h->x.p == a);
    EXPECT(btcx::guard([] { btcx::fail(BTC_ERR_HIP, "failed"); }) == BTC_ERR_HIP);
    btcx::free_handle(h);
    EXPECT(waits == 1);
    h = make(stream(4));
    EXPECT(h->x.p == a);
    btcx::free_handle(h);
    EXPECT(waits == 1);
    // a handle that a failing call drops: its work may be pending
    EXPECT(btcx::guard([] {
               std::unique_ptr<Handle> x(make(stream(5)));
               btcx::fail(BTC_ERR_ARG, "half-way");
           }) == BTC_ERR_ARG);
    h = make(stream(6));
    EXPECT(h->x.p != a && waits == 1);
    btcx::free_handle(h);  // settles what the failing call left
    EXPECT(waits == 2);
}

// A call's buffers, released in order on its stream, are idle once the call
// has waited for the stream -- not those that another thread released on it
// after that wait began.
void waited_streams() {
    void* a = pool_alloc(1 << 16, true, stream(1));
    pool_free(a, true, stream(1));
    during_sync = [] {
        void* b = pool_alloc(1 << 18, true, stream(1));
        pool_free(b, true, stream(1));
    };
    btcx::stream_wait(stream(1));
    during_sync = nullptr;
    void* c = pool_alloc(1 << 16, true, stream(2));
    EXPECT(c == a && waits == 0);
    const int before = mallocs;
    void* d = pool_alloc(1 << 18, true, stream(2));
    EXPECT(mallocs == before + 1 && waits == 0);
    pool_free(c, true, stream(2));
    pool_free(d, true, stream(2));
    // the per-thread handle: another thread's wait says nothing about this one's stream
    void* e = pool_alloc(1 << 20, true, hipStreamPerThread);
    pool_free(e, true, hipStreamPerThread);
    on_thread([] { btcx::stream_wait(hipStreamPerThread); });
    void* f = pool_alloc(1 << 20, true, stream(2));
    EXPECT(f != e);
    btcx::stream_wait(hipStreamPerThread);
    void* g = pool_alloc(1 << 20, true, stream(2));
    EXPECT(g == e);
    pool_free(f, true, stream(2));
    pool_free(g, true, stream(2));
}

// The cache is bounded in bytes and in blocks, and no call gives back more
// than a few blocks beyond what it brings; larger blocks are not kept.
void bounded() {
    std::vector<void*> p;
    for (int k = 0; k < 20000; ++k) p.push_back(pool_alloc(512, true, stream(1)));
    int most = 0;
    for (void* x : p) {
        const int before = frees;
        pool_free(x, true, stream(1));
        most = std::max(most, frees - before);
    }
    EXPECT(blocks.size() <= 5000 && most <= 2);
    p.clear();
    for (int k = 0; k < 24; ++k) p.push_back(pool_alloc(size_t(1) << 30, true, stream(1)));
    for (void* x : p) pool_free(x, true, stream(1));
    EXPECT(in_use <= (size_t(8) << 30));
    void* big = pool_alloc(size_t(5) << 30, true, stream(1));
    const int before = frees;
    pool_free(big, true, stream(1));
    EXPECT(frees == before + 1);
    // a refused allocation returns the cache and is tried again
    capacity = size_t(9) << 30;
    void* x = pool_alloc(size_t(8) << 30, true, stream(2));
    EXPECT(x && in_use == (size_t(8) << 30));
    EXPECT(btcx::guard([] { pool_alloc(size_t(2) << 30, true, stream(2)); }) == BTC_ERR_NOMEM);
    pool_free(x, true, stream(2));
    EXPECT(in_use == 0);
}

// The block that wastes least, at most an eighth (twice for small ones), and
// the newest of its size that may be used.
void sizes() {
    const size_t kSizes[] = {1 << 20, (1 << 20) + (1 << 17), (1 << 20) + (1 << 18)};
    std::map<size_t, void*> at;
    for (size_t b : kSizes) at[b] = pool_alloc(b, true, stream(1));
    for (size_t b : kSizes) pool_free(at[b], true, stream(1));
    for (int k = 0; k < 3; ++k)
        for (size_t b : kSizes) {
            void* p = pool_alloc(b - 100, true, stream(1));
            EXPECT(p == at[b]);
            pool_free(p, true, stream(1));
        }
    void* p = pool_alloc(1 << 20, true, stream(1));
    void* q = pool_alloc(1 << 20, true, stream(1));  // an eighth more
    const int before = mallocs;
    void* r = pool_alloc(1 << 20, true, stream(1));  // a quarter more is left
    EXPECT(p == at[kSizes[0]] && q == at[kSizes[1]] && mallocs == before + 1);
    pool_free(p, true, stream(1));
    pool_free(r, true, stream(1));
    pool_free(q, true, stream(2));  // another stream's
    EXPECT(pool_alloc(1 << 20, true, stream(1)) == r);
    EXPECT(pool_alloc(1 << 20, true, stream(1)) == p);
}

// What the cache holds goes back on request, handed-out blocks stay.
void trim() {
    void* a = pool_alloc(1 << 20, true, stream(1));
    void* b = pool_alloc(3 << 20, true, stream(2));
    void* c = pool_alloc(5 << 20, false, nullptr);
    pool_free(a, true, stream(1));
    pool_free(c, false, nullptr);
    int64_t bytes = -1;
    EXPECT(btc_memory_trim(&bytes) == BTC_OK && bytes == int64_t(6) << 20 && in_use == size_t(3) << 20);
    EXPECT(btc_memory_trim(nullptr) == BTC_OK && btc_memory_trim(&bytes) == BTC_OK && bytes == 0);
    pool_free(b, true, stream(2));
    EXPECT(pool_alloc(3 << 20, true, stream(2)) == b);
}

// Per-vertex sums of a count that has been waited for serve the next count on
// any stream; those of a count that failed do not before a wait.
void count_sums() {
    void* first = nullptr;
    for (int k = 1; k <= 5; ++k) {
        btcx::PvBuf pv;
        pv.alloc_on(1 << 16, k, stream(k));
        if (!first) first = pv.data();
        EXPECT(pv.data() == first);
        pv.release_idle();
    }
    EXPECT(mallocs == 1 && waits == 0);
    EXPECT(btcx::guard([] {
               btcx::PvBuf pv;
               pv.alloc_on(1 << 16, 1, stream(1));
               btcx::fail(BTC_ERR_HIP, "failed");
           }) == BTC_ERR_HIP);
    btcx::PvBuf pv;
    pv.alloc_on(1 << 16, 1, stream(1));
    EXPECT(mallocs == 2 && waits == 0);
    pv.release_idle();
    EXPECT(waits == 1);
}

const struct {
    const char* name;
    void (*run)();
} kChecks[] = {
    {"per_thread_stream", per_thread_stream},
    {"no_waits", no_waits},
    {"handles", handles},
    {"waited_streams", waited_streams},
    {"bounded", bounded},
    {"sizes", sizes},
    {"trim", trim},
    {"count_sums", count_sums},
};

}  // namespace

int main(int argc, char** argv) {
    for (const auto& c : kChecks)
        if (argc == 2 && std::string(argv[1]) == c.name) {
            c.run();
            if (!failures) std::puts("pool ok");
            return failures != 0;
        }
    std::fprintf(stderr, "usage: pool_check CHECK\n");
    return 2;
}
