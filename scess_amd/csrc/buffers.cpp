#include "buffers.h"

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>

namespace scess {

// ------------------------------------------------------------------- blocks
namespace {

// The caches of the process; left alone at its end
std::mutex g_caches_mu;
std::vector<BlockCache *> &g_caches = *new std::vector<BlockCache *>;

// What was freed on the runtime's side goes back to the device
void trim_pool(int device) {
    hipMemPool_t pool;
    if (hipDeviceGetDefaultMemPool(&pool, device) == hipSuccess)
        (void)hipMemPoolTrimTo(pool, 0);
    (void)hipGetLastError();
}

}  // namespace

BlockCache::BlockCache() {
    std::lock_guard<std::mutex> lk(g_caches_mu);
    g_caches.push_back(this);
}

BlockCache::~BlockCache() {
    {
        std::lock_guard<std::mutex> lk(g_caches_mu);
        g_caches.erase(std::find(g_caches.begin(), g_caches.end(), this));
    }
    flush();
}

// A block of this cache, or one of the runtime
hipError_t BlockCache::take(void **p, size_t bytes, hipStream_t s) {
    try {  // put() must not have to allocate
        used_.reserve(used_.size() + 1);
        free_.reserve(free_.size() + used_.size() + 1);
    } catch (...) {
        return hipErrorOutOfMemory;
    }
    // the smallest kept block that wastes at most half of itself (64 KiB of a small one)
    size_t best = free_.size();
    for (size_t i = 0; i < free_.size(); i++)
        if (free_[i].s == s && free_[i].bytes >= bytes && free_[i].bytes <= std::max<size_t>(2 * bytes, 65536) &&
            (best == free_.size() || free_[i].bytes < free_[best].bytes))
            best = i;
    if (best < free_.size()) {
        used_.push_back(free_[best]);
        cached_ -= free_[best].bytes;
        free_[best] = free_.back();
        free_.pop_back();
        *p = used_.back().p;
        return hipSuccess;
    }
    if (device_ < 0)
        (void)hipGetDevice(&device_);
    const hipError_t e = hipMallocAsync(p, bytes, s);
    if (e == hipSuccess)
        used_.push_back({*p, bytes, s});
    else
        *p = nullptr;
    return e;
}

hipError_t BlockCache::get(void **p, size_t bytes, hipStream_t s) {
    bytes = (std::max<size_t>(bytes, 16) + 255) / 256 * 256;
    *p = nullptr;
    hipError_t e = take(p, bytes, s);
    if (e == hipErrorOutOfMemory) {
        // what is missing may be kept here or by another context, or freed but still with the runtime's pool
        (void)hipGetLastError();
        (void)hipStreamSynchronize(s);
        trim_all(device_);
        e = take(p, bytes, s);
    }
    return e;
}

void BlockCache::put(void *p) {
    if (!p)
        return;
    for (size_t i = used_.size(); i-- > 0;)
        if (used_[i].p == p) {
            const Block b = used_[i];
            used_[i] = used_.back();
            used_.pop_back();
            if (cached_ + b.bytes <= kMaxCached) {
                free_.push_back(b);
                cached_ += b.bytes;
            } else {
                (void)hipFreeAsync(b.p, b.s);
            }
            return;
        }
}

void BlockCache::flush() {
    for (const Block &b : free_)
        (void)hipFreeAsync(b.p, b.s);
    free_.clear();
    cached_ = 0;
}

void BlockCache::trim() {
    if (device_ < 0)
        return;
    hipStream_t last = nullptr;
    for (const Block &b : free_) {
        (void)hipFreeAsync(b.p, b.s);
        if (last && b.s != last)
            (void)hipStreamSynchronize(last);
        last = b.s;
    }
    if (last)
        (void)hipStreamSynchronize(last);
    free_.clear();
    cached_ = 0;
    trim_pool(device_);
}

// A context ends in a Use that flushes, before its streams go, and leaves the list before its cache does: what is found here
// has its stream or no blocks
void BlockCache::trim_all(int device) {
    std::lock_guard<std::mutex> lk(g_caches_mu);
    for (BlockCache *c : g_caches) {
        std::unique_lock<std::recursive_mutex> use(c->use_, std::try_to_lock);
        if (use.owns_lock() && c->device_ == device)
            c->trim();
    }
}

// ------------------------------------------------------------------- copies
namespace {

constexpr size_t kChunk = (size_t)2 << 20, kPiece = (size_t)1 << 19;
constexpr int kSlots = 8, kThreads = 6, kPieces = kSlots * (int)(kChunk / kPiece);
constexpr size_t kLarge = (size_t)4 << 20;  // below it the runtime's own staging is as good
// Pinned memory and threads take 2 ms to set up, which some 40 MB of copies gain: made once larger copies add up to this
constexpr size_t kWorthIt = (size_t)64 << 20;

// Threads that carry out memcpy pieces; a batch is a counter of the pieces still to do
struct Ring {
    char *pinned = nullptr;
    std::mutex use;  // one copy at a time
    std::mutex m;
    std::condition_variable work, done;
    struct Piece {
        char *dst;
        const char *src;
        size_t n;
        int *left;
    };
    Piece queue[kPieces];  // circular; a slot is started again only after its pieces are done
    unsigned head = 0, tail = 0;
    Piece pop() { return queue[head++ % kPieces]; }
    bool stop = false;
    std::vector<std::thread> threads;

    ~Ring() {
        {
            std::lock_guard<std::mutex> lk(m);
            stop = true;
        }
        work.notify_all();
        for (auto &t : threads)
            t.join();
        if (pinned)
            (void)hipHostFree(pinned);
    }
    size_t copied = 0;
    bool ready(size_t bytes) {
        if (pinned)
            return true;
        if ((copied += bytes) < kWorthIt)
            return false;
        if (hipHostMalloc((void **)&pinned, kChunk * kSlots, hipHostMallocPortable) != hipSuccess) {
            (void)hipGetLastError();
            pinned = nullptr;
            return false;
        }
        try {
            for (int i = 0; i < kThreads; i++)
                threads.emplace_back([this] { loop(); });
        } catch (...) {  // fewer threads, or none: wait() helps out
        }
        return true;
    }
    static void finish(Ring &r, const Piece &p, std::unique_lock<std::mutex> &lk) {
        lk.unlock();
        std::memcpy(p.dst, p.src, p.n);
        lk.lock();
        if (--*p.left == 0)
            r.done.notify_all();
    }
    void loop() {
        std::unique_lock<std::mutex> lk(m);
        while (true) {
            work.wait(lk, [this] { return stop || head != tail; });
            if (head == tail)
                return;
            const Piece p = pop();
            finish(*this, p, lk);
        }
    }
    void start(char *dst, const char *src, size_t n, int *left) {
        {
            std::lock_guard<std::mutex> lk(m);
            *left = (int)((n + kPiece - 1) / kPiece);
            for (size_t o = 0; o < n; o += kPiece)
                queue[tail++ % kPieces] = {dst + o, src + o, std::min(kPiece, n - o), left};
        }
        work.notify_all();
    }
    void wait(int *left) {
        std::unique_lock<std::mutex> lk(m);
        while (*left > 0) {
            if (head != tail) {
                const Piece p = pop();
                finish(*this, p, lk);
            } else {
                done.wait(lk, [&] { return *left == 0 || head != tail; });
            }
        }
    }
};

std::mutex g_ring_mu;
int g_ring_users = 0;
std::shared_ptr<Ring> &g_ring = *new std::shared_ptr<Ring>;  // left alone at the end of the process

std::shared_ptr<Ring> ring() {
    std::lock_guard<std::mutex> lk(g_ring_mu);
    return g_ring;
}

}  // namespace

void copies_retain() {
    std::lock_guard<std::mutex> lk(g_ring_mu);
    if (g_ring_users++ == 0) {
        try {
            g_ring = std::make_shared<Ring>();
        } catch (...) {  // copies then go the plain way
        }
    }
}

void copies_release() {
    std::shared_ptr<Ring> last;  // ends outside the lock
    std::lock_guard<std::mutex> lk(g_ring_mu);
    if (--g_ring_users == 0)
        last.swap(g_ring);
}

// Chunks i of the copy use slot i % kSlots; per slot the event of its device copy and the pieces of its host copy
static hipError_t ring_copy(Ring &r, char *h, char *d, size_t bytes, hipStream_t s, bool down) {
    const size_t n = (bytes + kChunk - 1) / kChunk;
    hipEvent_t ev[kSlots] = {};
    int left[kSlots] = {};
    hipError_t e = hipSuccess;
    for (int i = 0; i < kSlots && e == hipSuccess; i++)
        e = hipEventCreateWithFlags(&ev[i], hipEventDisableTiming);
    auto len = [&](size_t i) { return std::min(kChunk, bytes - i * kChunk); };
    auto slot = [&](size_t i) { return r.pinned + (i % kSlots) * kChunk; };
    // `first` is the leading side (device copies down, host copies up), `second` follows it chunk by chunk
    size_t led = 0;
    for (size_t i = 0; i < n && e == hipSuccess; i++) {
        for (; led < n && led < i + kSlots && e == hipSuccess; led++) {
            const int q = (int)(led % kSlots);
            if (down) {
                r.wait(&left[q]);  // the slot's last chunk is out
                e = hipMemcpyAsync(slot(led), d + led * kChunk, len(led), hipMemcpyDeviceToHost, s);
                if (e == hipSuccess)
                    e = hipEventRecord(ev[q], s);
            } else {
                if (led >= kSlots)
                    e = hipEventSynchronize(ev[q]);
                if (e == hipSuccess)
                    r.start(slot(led), h + led * kChunk, len(led), &left[q]);
            }
        }
        if (e != hipSuccess)
            break;
        const int q = (int)(i % kSlots);
        if (down) {
            e = hipEventSynchronize(ev[q]);
            if (e == hipSuccess)
                r.start(h + i * kChunk, slot(i), len(i), &left[q]);
        } else {
            r.wait(&left[q]);
            e = hipMemcpyAsync(d + i * kChunk, slot(i), len(i), hipMemcpyHostToDevice, s);
            if (e == hipSuccess)
                e = hipEventRecord(ev[q], s);
        }
    }
    if (e != hipSuccess)  // nothing may still be writing or reading the ring
        (void)hipStreamSynchronize(s);
    for (int i = 0; i < kSlots; i++) {
        r.wait(&left[i]);
        if (ev[i]) {
            if (!down)  // the ring is free for the next copy once the device has read it
                (void)hipEventSynchronize(ev[i]);
            (void)hipEventDestroy(ev[i]);
        }
    }
    return e;
}

// Pinned and managed host memory is copied directly (the ring would only add a copy), and device memory has to be
static bool pageable(const void *h) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, h) == hipSuccess)
        return a.type == hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return true;
}

hipError_t copy_to_host(void *h, const void *d, size_t bytes, hipStream_t s) {
    if (bytes >= kLarge && pageable(h)) {
        if (const std::shared_ptr<Ring> r = ring()) {
            std::unique_lock<std::mutex> lk(r->use, std::try_to_lock);  // in use by another thread: the plain way
            if (lk.owns_lock() && r->ready(bytes))
                return ring_copy(*r, (char *)h, (char *)d, bytes, s, true);
        }
    }
    hipError_t e = hipMemcpyAsync(h, d, bytes, hipMemcpyDeviceToHost, s);
    return e == hipSuccess ? hipStreamSynchronize(s) : e;
}

hipError_t copy_to_device(void *d, const void *h, size_t bytes, hipStream_t s) {
    if (bytes >= kLarge && pageable(h)) {
        if (const std::shared_ptr<Ring> r = ring()) {
            std::unique_lock<std::mutex> lk(r->use, std::try_to_lock);  // in use by another thread: the plain way
            if (lk.owns_lock() && r->ready(bytes))
                return ring_copy(*r, (char *)h, (char *)d, bytes, s, false);
        }
    }
    return hipMemcpyAsync(d, h, bytes, hipMemcpyHostToDevice, s);
}

}  // namespace scess
