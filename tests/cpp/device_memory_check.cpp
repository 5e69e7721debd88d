// Checks of xitils_amd/csrc/device_memory.h on the host stand-in for HIP.
#include "../../xitils_amd/csrc/device_memory.h"

#include <cstdio>
#include <thread>

#define CHECK(c)                                                   \
    do {                                                           \
        if (!(c)) {                                                \
            std::printf("FAIL line %d: %s\n", __LINE__, #c);       \
            return 1;                                              \
        }                                                          \
    } while (0)

constexpr size_t MB = (size_t)1 << 20;

int main() {
    {
        StagePool pool(0), second(0), other(1);
        // a kept block serves the next call
        void *a = nullptr, *b = nullptr;
        CHECK(pool.take(40 * MB, &a) == hipSuccess);
        pool.give(a);
        CHECK(pool.take(30 * MB, &b) == hipSuccess && b == a);
        pool.give(b);
        CHECK(fake.used[0] == 40 * MB && fake.mallocs == 1);
        // no more than KEEP is held
        CHECK(pool.take(100 * MB, &a) == hipSuccess && fake.used[0] == 100 * MB);
        pool.give(a);
        CHECK(pool.take(StagePool::KEEP + MB, &a) == hipSuccess && fake.used[0] == StagePool::KEEP + MB);
        pool.give(a);
        CHECK(fake.used[0] == 0);
        // another allocation that runs out of memory gets what the GPU's pools
        // keep, not what is in use and not the other GPU's
        void *used = nullptr, *kept = nullptr;
        CHECK(pool.take(50 * MB, &used) == hipSuccess && pool.take(60 * MB, &kept) == hipSuccess);
        pool.give(kept);
        CHECK(second.take(70 * MB, &kept) == hipSuccess);
        second.give(kept);
        fake_device = 1;
        CHECK(other.take(20 * MB, &kept) == hipSuccess);
        other.give(kept);
        fake_device = 0;
        float* x = nullptr;
        CHECK(dalloc(&x, 200 * MB / sizeof(float)) == hipSuccess && x);
        CHECK(fake.used[0] == 250 * MB && fake.used[1] == 20 * MB);
        CHECK(hipGetLastError() == hipSuccess);
        float* y = nullptr;   // nothing is kept any more
        CHECK(dalloc(&y, 10 * MB / sizeof(float)) == hipErrorOutOfMemory && !y);
        CHECK(hipGetLastError() == hipErrorOutOfMemory);
        CHECK(second.take(7 * MB, &kept) == hipErrorOutOfMemory);
        (void)hipGetLastError();
        CHECK(hipFree(x) == hipSuccess);
        pool.give(used);
        CHECK(dalloc(&y, 0) == hipSuccess && !y);
        // several threads take, give and run out of memory
        auto work = [&](StagePool& p, unsigned seed) {
            for (int i = 0; i < 4000; ++i) {
                seed = seed * 1664525u + 1013904223u;
                void* v = nullptr;
                if (seed & 0x10000u) {
                    if (p.take(MB + (seed >> 20) * 20000, &v) == hipSuccess) p.give(v);
                } else if (device_malloc(&v, 90 * MB) == hipSuccess) {
                    hipFree(v);
                }
            }
        };
        std::thread t[4];
        for (unsigned k = 0; k < 4; ++k) t[k] = std::thread(work, std::ref(k & 1 ? second : pool), k);
        for (std::thread& k : t) k.join();
        CHECK(fake.used[0] <= 2 * StagePool::KEEP);
    }
    CHECK(fake.live.empty() && fake.used[0] == 0 && fake.used[1] == 0);
    std::printf("OK\n");
    return 0;
}
