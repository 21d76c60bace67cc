// Device blocks kept by a context between calls, and copies between pageable host memory and the device.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>
#include <vector>

namespace scess {

// Device memory of one context: freed blocks are kept, up to kMaxCached bytes in all, and handed out again; the rest goes
// back to the runtime, and everything at the end of the context, on trim(), and where a context of the process finds the
// device full. Stream ordered: a block is reused by work on the same stream (or ordered after it). A call's dozens of
// allocations otherwise cost more than its kernels for small systems, and the mapping of freshly allocated memory some
// milliseconds per GiB for large ones. Whoever uses it holds a Use for the length of the call; another thread only frees the
// blocks of a context that is not in a call (trim_all).
class BlockCache {
public:
    static constexpr size_t kMaxCached = (size_t)6 << 30;
    BlockCache();
    ~BlockCache();
    BlockCache(const BlockCache &) = delete;
    BlockCache &operator=(const BlockCache &) = delete;
    struct Use {  // (a callback out of a call may make another one on the same context)
        explicit Use(BlockCache &c) : lk(c.use_) {}
        std::lock_guard<std::recursive_mutex> lk;
    };
    hipError_t get(void **p, size_t bytes, hipStream_t s);
    void put(void *p);  // null is allowed
    void flush();       // the kept blocks go back to the runtime, in the order of their streams
    void trim();        // the kept blocks go back to the device, once the work that used them is done
    // p to at least `need` elements, without its contents; after an error p is null and cap 0
    template <class T> hipError_t grow(T *&p, size_t &cap, size_t need, hipStream_t s) {
        if (need <= cap)
            return hipSuccess;
        put((void *)p);
        p = nullptr;
        cap = 0;
        const hipError_t e = get((void **)&p, sizeof(T) * need, s);
        if (e == hipSuccess)
            cap = need;
        return e;
    }

private:
    struct Block {
        void *p;
        size_t bytes;
        hipStream_t s;
    };
    hipError_t take(void **p, size_t bytes, hipStream_t s);
    static void trim_all(int device);  // of every context on the device that is not in a call, and of this thread's
    std::recursive_mutex use_;
    std::vector<Block> free_, used_;
    size_t cached_ = 0;
    int device_ = -1;  // of the blocks; -1 before the first
};

// Copies of any size between host memory and the device, ordered on stream s as hipMemcpyAsync would be. Large ones of
// pageable memory go through a ring of pinned chunks shared by the process, filled or emptied by a few threads: one
// thread's memcpy (and its page faults in a new array) runs at 5-13 GB/s, the link at 50 (gradients of o=20, v=200 to the
// host, 1.6 GB: 100 ms -> 30; transform of 58 functions, 91 MB each way: 14.7 -> 9.6). copy_to_host returns when the data
// is there; copy_to_device when a pageable `h` has been read.
hipError_t copy_to_host(void *h, const void *d, size_t bytes, hipStream_t s);
hipError_t copy_to_device(void *d, const void *h, size_t bytes, hipStream_t s);
// The ring and its threads exist while a context does
void copies_retain();
void copies_release();

}  // namespace scess
