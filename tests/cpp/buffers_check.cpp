// Host-only check of the device block cache and the copy ring (scess_amd/csrc/buffers.cpp) over a simulated device: the
// HIP calls that buffers.cpp makes are defined here. Copies are carried out as late as the waits allow. Memory is a count of bytes with a limit; a freed block goes to the pool when its
// stream is next waited for, and back to the device when the pool is trimmed. Run by tests/test_buffers_cpu.py with the name of one check.
#include "buffers.h"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <thread>
#include <utility>
#include <vector>

namespace {

struct Device {
    size_t limit = (size_t)1 << 40, held = 0, pool = 0;  // bytes of the device, taken from it, and of these in the pool
    std::map<void *, size_t> live, freed;                // by address: nothing is behind it
    size_t next = 4096;
    std::vector<std::function<void()>> queue;  // of the only stream that copies
    size_t done = 0;                           // of them
    std::vector<size_t> copies;                // their sizes
    const void *pinned = nullptr;              // host memory that the caller allocated as pinned
    size_t ring = 0;                           // bytes of pinned memory held
    void run(size_t n) {
        for (; done < n; done++)
            queue[done]();
    }
} dev;

}  // namespace

extern "C" {
hipError_t hipMallocAsync(void **p, size_t bytes, hipStream_t) {
    if (dev.held + bytes > dev.limit)
        return hipErrorOutOfMemory;
    *p = (void *)dev.next;
    dev.next += (bytes + 4095) / 4096 * 4096;
    dev.held += bytes;
    dev.live[*p] = bytes;
    return hipSuccess;
}
hipError_t hipFreeAsync(void *p, hipStream_t) {
    const auto it = dev.live.find(p);
    if (it == dev.live.end())
        return hipErrorInvalidValue;
    dev.freed.insert(*it);
    dev.live.erase(it);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    dev.run(dev.queue.size());
    for (auto &f : dev.freed)
        dev.pool += f.second;
    dev.freed.clear();
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t *p, int) {
    *p = nullptr;
    return hipSuccess;
}
hipError_t hipMemPoolTrimTo(hipMemPool_t, size_t) {
    dev.held -= dev.pool;
    dev.pool = 0;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned int) {
    *p = std::malloc(bytes);
    std::memset(*p, 0xff, bytes);
    dev.ring = bytes;
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    std::free(p);
    dev.ring = 0;
    return hipSuccess;
}
// an event is the number of operations before it
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = (hipEvent_t) new size_t(0);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    *(size_t *)e = dev.queue.size();
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    dev.run(*(size_t *)e);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    delete (size_t *)e;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    dev.copies.push_back(n);
    dev.queue.push_back([=] { std::memcpy(d, s, n); });
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
    a->type = dev.pinned && p == dev.pinned ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return hipSuccess;
}
}

#define REQUIRE(x)                                             \
    do {                                                       \
        if (!(x)) {                                            \
            std::printf("line %d: %s is false\n", __LINE__, #x); \
            std::exit(1);                                      \
        }                                                      \
    } while (0)

static hipStream_t stream(int n = 1) { return (hipStream_t)(size_t)(16 * n); }

// A growth that fails leaves a null pointer of no capacity, so the next call does not use it; a smaller need then works
static void grow() {
    dev.limit = 1 << 20;
    scess::BlockCache c;
    double *p = nullptr;
    size_t cap = 0;
    REQUIRE(c.grow(p, cap, 1000, stream()) == hipSuccess && p && cap == 1000);
    double *const first = p;
    REQUIRE(c.grow(p, cap, 500, stream()) == hipSuccess && p == first && cap == 1000);
    REQUIRE(c.grow(p, cap, 1 << 20, stream()) == hipErrorOutOfMemory);
    REQUIRE(!p && cap == 0);
    REQUIRE(c.grow(p, cap, 1000, stream()) == hipSuccess && p && cap == 1000);
    c.put(p);
}

// A block past the cache's bound goes back to the runtime, which may still hold it when a larger one is asked for
static void freed_block_in_pool() {
    const size_t gib = (size_t)1 << 30;
    dev.limit = 20 * gib;
    scess::BlockCache c;
    void *p = nullptr, *q = nullptr;
    REQUIRE(c.get(&p, 8 * gib, stream()) == hipSuccess);
    c.put(p);  // nothing is kept of it
    REQUIRE(c.get(&q, 16 * gib, stream()) == hipSuccess && q);
    c.put(q);
    // kept blocks make room, too
    REQUIRE(c.get(&p, 5 * gib, stream()) == hipSuccess);
    c.put(p);
    REQUIRE(c.get(&q, 18 * gib, stream()) == hipSuccess && q);
    c.put(q);
    REQUIRE(c.get(&q, 21 * gib, stream()) == hipErrorOutOfMemory && !q);
}

// Blocks that one context keeps make room for another, and trim() gives them back
static void other_contexts() {
    const size_t gib = (size_t)1 << 30;
    dev.limit = 10 * gib;
    scess::BlockCache a, b;
    void *p = nullptr, *q = nullptr, *r = nullptr;
    REQUIRE(a.get(&p, 5 * gib, stream(1)) == hipSuccess && a.get(&r, gib, stream(1)) == hipSuccess);
    a.put(p);
    REQUIRE(b.get(&q, 8 * gib, stream(2)) == hipSuccess && q);
    REQUIRE(dev.live.count(r) == 1 && dev.live.size() == 2);  // what is in use stays
    b.put(q);
    REQUIRE(a.get(&p, gib, stream(1)) == hipSuccess);
    a.put(p);
    a.put(r);
    REQUIRE(dev.held >= 2 * gib);
    a.trim();
    REQUIRE(dev.held == 0 && dev.live.empty());
    a.trim();
    // not those of a context in a call on another thread
    REQUIRE(a.get(&p, 5 * gib, stream(1)) == hipSuccess && p);
    a.put(p);
    hipError_t e = hipSuccess;
    {
        const scess::BlockCache::Use use(a);
        std::thread([&] { e = b.get(&q, 8 * gib, stream(2)); }).join();
    }
    REQUIRE(e == hipErrorOutOfMemory && !q);
    std::thread([&] { e = b.get(&q, 8 * gib, stream(2)); }).join();
    REQUIRE(e == hipSuccess && q);
    b.put(q);
}

static std::vector<char> bytes(size_t n, unsigned seed) {
    std::vector<char> x(n);
    for (auto &b : x) {
        seed = seed * 1664525u + 1013904223u;
        b = (char)(seed >> 24);
    }
    return x;
}

// More than the 64 MiB of large copies after which the ring is made
static void start_ring() {
    const std::vector<char> x = bytes((size_t)40 << 20, 1);
    std::vector<char> y(x.size());
    for (int i = 0; i < 2; i++) {
        REQUIRE(scess::copy_to_device(y.data(), x.data(), x.size(), stream()) == hipSuccess);
        REQUIRE(hipStreamSynchronize(stream()) == hipSuccess && y == x);
    }
    REQUIRE(dev.ring > 0);
}

// Both ways, at the edges of chunks (2 MiB) and slots (8): pieces go through the ring, and every byte arrives
static void ring() {
    scess::copies_retain();
    start_ring();
    const size_t mib = (size_t)1 << 20;
    for (size_t n : {4 * mib, 4 * mib + 1, 6 * mib - 1, 6 * mib, 8 * mib, 16 * mib - 8, 16 * mib, 16 * mib + 8, 18 * mib,
                     33 * mib + 12345})
        for (int down = 0; down < 2; down++) {
            const std::vector<char> x = bytes(n, (unsigned)n);
            std::vector<char> y(n, 0);
            dev.copies.clear();
            if (down) {
                REQUIRE(scess::copy_to_host(y.data(), x.data(), n, stream()) == hipSuccess);
            } else {
                std::vector<char> h = x;
                REQUIRE(scess::copy_to_device(y.data(), h.data(), n, stream()) == hipSuccess);
                h.assign(n, 0);  // has been read
                REQUIRE(hipStreamSynchronize(stream()) == hipSuccess);
            }
            REQUIRE(y == x);
            REQUIRE(dev.copies.size() == (n + 2 * mib - 1) / (2 * mib));
        }
    scess::copies_release();
    REQUIRE(dev.ring == 0);
}

// Memory that the caller has pinned is copied in one piece, without the ring
static void pinned() {
    scess::copies_retain();
    start_ring();
    std::vector<char> h = bytes((size_t)20 << 20, 7), d(h.size());
    dev.pinned = h.data();
    dev.copies.clear();
    REQUIRE(scess::copy_to_device(d.data(), h.data(), h.size(), stream()) == hipSuccess);
    REQUIRE(hipStreamSynchronize(stream()) == hipSuccess && d == h);
    REQUIRE(dev.copies.size() == 1 && dev.copies[0] == h.size());
    d = bytes(d.size(), 8);
    REQUIRE(scess::copy_to_host(h.data(), d.data(), h.size(), stream()) == hipSuccess && d == h);
    REQUIRE(dev.copies.size() == 2 && dev.copies[1] == h.size());
    scess::copies_release();
}

int main(int argc, char **argv) {
    const std::map<std::string, void (*)()> checks = {{"grow", grow},
                                                               {"freed_block_in_pool", freed_block_in_pool},
                                                               {"other_contexts", other_contexts},
                                                               {"ring", ring},
                                                               {"pinned", pinned}};
    const auto it = argc == 2 ? checks.find(argv[1]) : checks.end();
    if (it == checks.end())
        return 2;
    it->second();
    std::printf("ok\n");
    return 0;
}
