// Host stand-in for the few HIP calls of xitils_amd/csrc/device_memory.h: GPUs
// with FAKE_BYTES of memory each.
#pragma once

#include <cstddef>
#include <cstdlib>
#include <map>
#include <mutex>
#include <utility>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };

constexpr size_t FAKE_BYTES = (size_t)256 << 20;
struct FakeHip {
    std::mutex mu;
    std::map<void*, std::pair<int, size_t>> live;
    size_t used[2] = {0, 0};
    int mallocs = 0;
};
inline FakeHip fake;
inline thread_local int fake_device = 0;
inline thread_local hipError_t fake_last = hipSuccess;

inline hipError_t hipGetDevice(int* d) {
    *d = fake_device;
    return hipSuccess;
}
inline hipError_t hipGetLastError() { return std::exchange(fake_last, hipSuccess); }
inline hipError_t hipMalloc(void** p, size_t bytes) {
    std::lock_guard<std::mutex> lock(fake.mu);
    if (fake.used[fake_device] + bytes > FAKE_BYTES) {
        *p = nullptr;
        return fake_last = hipErrorOutOfMemory;
    }
    *p = std::malloc(1);
    fake.live[*p] = {fake_device, bytes};
    fake.used[fake_device] += bytes;
    fake.mallocs++;
    return hipSuccess;
}
inline hipError_t hipFree(void* p) {
    if (!p) return hipSuccess;
    std::lock_guard<std::mutex> lock(fake.mu);
    auto it = fake.live.find(p);
    if (it == fake.live.end()) return fake_last = hipErrorInvalidValue;
    fake.used[it->second.first] -= it->second.second;
    fake.live.erase(it);
    std::free(p);
    return hipSuccess;
}
