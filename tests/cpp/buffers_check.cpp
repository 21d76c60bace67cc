// Host-only check of the device block cache (scess_amd/csrc/buffers.cpp) over a simulated device: the HIP calls that
// buffers.cpp makes are defined here. Memory is a count of bytes with a limit; a freed block goes to the pool when its
// stream is next waited for, and back to the device when the pool is trimmed. Run by tests/test_buffers_cpu.py with the name of one check.
#include "buffers.h"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {

struct Device {
    size_t limit = (size_t)1 << 40, held = 0, pool = 0;  // bytes of the device, taken from it, and of these in the pool
    std::map<void *, size_t> live, freed;                // by address: nothing is behind it
    size_t next = 4096;
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
hipError_t hipHostMalloc(void **, size_t, unsigned int) { return hipErrorOutOfMemory; }
hipError_t hipHostFree(void *) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *, unsigned) { return hipErrorUnknown; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipErrorUnknown; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) { return hipErrorUnknown; }
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
    REQUIRE(a.get(&p, gib, stream(1)) == hipSuccess && p);
    a.put(p);
}

int main(int argc, char **argv) {
    const std::map<std::string, void (*)()> checks = {{"grow", grow}, {"freed_block_in_pool", freed_block_in_pool},
                                                               {"other_contexts", other_contexts}};
    const auto it = argc == 2 ? checks.find(argv[1]) : checks.end();
    if (it == checks.end())
        return 2;
    it->second();
    std::printf("ok\n");
    return 0;
}
