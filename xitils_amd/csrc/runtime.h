// Host-side pieces shared by the library's translation units (runtime.hip,
// vmf.hip): the device handle, error reporting and allocation helpers.
#pragma once

#include <hip/hip_runtime.h>

#include <string>

#include "../../include/xitils_amd.h"

#include <mutex>

struct MultiState;   // unified-batch buffers (runtime.hip)
struct RenderPool;   // xt_render's path buffers, shared by the device's scenes (runtime.hip)

// Device memory for the copies of callers' host arrays, kept between calls: a
// hipMalloc and hipFree pair costs 100 us and more, and hipFree waits for the
// whole device (three calls on 96 vMF mixtures from host arrays: 3119 -> 2996 us).  At most KEEP bytes are held, given back with the device handle
// or when an allocation fails; what does not fit is freed when given back.
class StagePool {
public:
    static constexpr size_t KEEP = (size_t)128 << 20;
    hipError_t take(size_t bytes, void** p) {
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
        hipError_t e = hipMalloc(p, bytes);
        if (e == hipErrorOutOfMemory && held > 0) {
            (void)hipGetLastError();
            drop_free();
            e = hipMalloc(p, bytes);
        }
        if (e == hipSuccess && held + bytes <= KEEP)
            for (Block& b : blocks)
                if (!b.p) {
                    b = {*p, bytes, true};
                    held += bytes;
                    break;
                }
        return e;
    }
    // The caller's work on p has ended.
    void give(void* p) {
        if (!p) return;
        std::lock_guard<std::mutex> lock(mu);
        for (Block& b : blocks)
            if (b.p == p) {
                b.busy = false;
                return;
            }
        hipFree(p);
    }
    ~StagePool() {
        for (Block& b : blocks) hipFree(b.p);
    }

private:
    struct Block {
        void* p = nullptr;
        size_t bytes = 0;
        bool busy = false;
    };
    void drop_free() {
        for (Block& b : blocks)
            if (b.p && !b.busy) {
                held -= b.bytes;
                hipFree(b.p);
                b = Block{};
            }
    }
    std::mutex mu;
    Block blocks[64];
    size_t held = 0;
};

struct xt_device {
    int ordinal = 0;
    int num_cu = 0;
    std::string arch;
    MultiState* multi = nullptr;        // created by the first unified xt_render_batch
    RenderPool* pool = nullptr;         // created by the first xt_render
    std::mutex pool_mu;                 // guards creating `pool`
    StagePool stage;                    // copies of host arrays
    unsigned char* query_io = nullptr;      // pinned rays and results of small host queries
    unsigned char* query_io_dev = nullptr;  // the same memory's device address
    bool query_busy = false;                // in some thread's query
    std::mutex query_mu;                    // guards the three
    unsigned char* scratch = nullptr;   // this device's address of the static scratch array (xt_render_static)
};

// Records msg as this thread's last error (xt_last_error) and returns s.
xt_status xt_fail(xt_status s, const std::string& msg);

#define XT_HIP(call)                                                                                   \
    do {                                                                                               \
        hipError_t e_ = (call);                                                                        \
        if (e_ != hipSuccess)                                                                          \
            return xt_fail(XT_ERR_DEVICE, std::string(#call) + " failed: " + hipGetErrorString(e_));    \
    } while (0)

template <class T>
hipError_t dalloc(T** p, size_t count) {
    *p = nullptr;
    if (count == 0) return hipSuccess;
    return hipMalloc((void**)p, count * sizeof(T));
}
