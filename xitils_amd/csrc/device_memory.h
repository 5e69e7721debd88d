// Device allocation of the library and the memory that it keeps between calls.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>

// Device memory for the copies of callers' host arrays, kept between calls: a
// hipMalloc and hipFree pair costs 100 us and more, and hipFree waits for the
// whole device (three calls on 96 vMF mixtures from host arrays: 3119 -> 2996 us).
// At most KEEP bytes are held, given back with the device handle or when any
// allocation of the library on that GPU fails; what does not fit is freed when
// given back.
class StagePool {
public:
    static constexpr size_t KEEP = (size_t)128 << 20;
    explicit StagePool(int ordinal) : ordinal(ordinal) {
        std::lock_guard<std::mutex> lock(pools_mu);
        next = pools;
        pools = this;
    }
    ~StagePool() {
        {
            std::lock_guard<std::mutex> lock(pools_mu);
            StagePool** at = &pools;
            while (*at != this) at = &(*at)->next;
            *at = next;
        }
        for (Block& b : blocks) (void)hipFree(b.p);
    }
    StagePool(const StagePool&) = delete;
    StagePool& operator=(const StagePool&) = delete;

    hipError_t take(size_t bytes, void** p);
    // The caller's work on p has ended.
    void give(void* p) {
        if (!p) return;
        std::lock_guard<std::mutex> lock(mu);
        for (Block& b : blocks)
            if (b.p == p) {
                b.busy = false;
                return;
            }
        (void)hipFree(p);
    }

    // Frees what the pools of the current GPU keep and nobody uses; how much.
    static size_t free_kept() {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) return 0;
        size_t n = 0;
        std::lock_guard<std::mutex> lock(pools_mu);
        for (StagePool* s = pools; s; s = s->next)
            if (s->ordinal == dev) {
                std::lock_guard<std::mutex> own(s->mu);
                n += s->drop_free();
            }
        return n;
    }

private:
    struct Block {
        void* p = nullptr;
        size_t bytes = 0;
        bool busy = false;
    };
    // every pool of the process (taken before a pool's own mutex)
    static inline std::mutex pools_mu;
    static inline StagePool* pools = nullptr;
    StagePool* next = nullptr;
    size_t drop_free() {
        size_t n = 0;
        for (Block& b : blocks)
            if (b.p && !b.busy) {
                n += b.bytes;
                (void)hipFree(b.p);
                b = Block{};
            }
        held -= n;
        return n;
    }
    const int ordinal;
    std::mutex mu;
    Block blocks[64];
    size_t held = 0;
};

// hipMalloc; where it runs out of memory, once more without what the pools keep.
inline hipError_t device_malloc(void** p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory && StagePool::free_kept() > 0) {
        (void)hipGetLastError();
        e = hipMalloc(p, bytes);
    }
    return e;
}

inline hipError_t StagePool::take(size_t bytes, void** p) {
    {
        std::lock_guard<std::mutex> lock(mu);
        Block* best = nullptr;
        for (Block& b : blocks)
            if (b.p && !b.busy && b.bytes >= bytes && (!best || b.bytes < best->bytes)) best = &b;
        if (best) {
            best->busy = true;
            *p = best->p;
            return hipSuccess;
        }
        if (held + bytes > KEEP) drop_free();
    }
    const hipError_t e = device_malloc(p, bytes);
    if (e != hipSuccess) return e;
    std::lock_guard<std::mutex> lock(mu);
    if (held + bytes <= KEEP)
        for (Block& b : blocks)
            if (!b.p) {
                b = {*p, bytes, true};
                held += bytes;
                break;
            }
    return e;
}

template <class T>
hipError_t dalloc(T** p, size_t count) {
    *p = nullptr;
    if (count == 0) return hipSuccess;
    return device_malloc((void**)p, count * sizeof(T));
}
