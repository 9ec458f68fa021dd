// ArenaPool and device_malloc (csrc/arena_pool.hpp) on the stand-in devices of
// tests/cpp/fake_hip.  Prints one line a scenario for tests/test_arena_pool_cpu.py.
#include <cstdio>
#include <memory>

#include "../../mcrg_amd/csrc/arena_pool.hpp"

using namespace mcrg;

namespace {
// A server's life: its arena from the pool or the device, back at its end.
bool serve(ArenaPool &pool, size_t bytes)
{
    void *p = pool.take(bytes);
    if (!p && device_malloc(&p, bytes) != hipSuccess) return false;
    if (!pool.give(p, bytes)) (void)hipFree(p);
    return true;
}
void reset(size_t a, size_t b)
{
    g_hip.room[0] = a;
    g_hip.room[1] = b;
    g_hip.device = 0;
    g_hip.frees = 0;
    g_hip.last = hipSuccess;
}
}  // namespace

int main()
{
    {
        reset(100, 0);
        {
            ArenaPool pool(0);
            std::printf("newest");
            for (size_t bytes : {40, 30, 30, 40, 40}) {
                serve(pool, bytes);
                std::printf(" %zu:%d", 100 - g_hip.room[0], g_hip.frees);
            }
        }
        std::printf(" end %zu\n", 100 - g_hip.room[0]);
    }
    {
        const size_t big = ArenaPool::kMaxBytes + 1;
        reset(3 * big, 0);
        ArenaPool pool(0);
        serve(pool, 7);
        serve(pool, big);
        std::printf("bounded %zu", 3 * big - g_hip.room[0]);
        serve(pool, ArenaPool::kMaxBytes);
        std::printf(" %d\n", 3 * big - g_hip.room[0] == ArenaPool::kMaxBytes);
    }
    {
        // an allocation that finds no memory: idle arenas of every context on
        // its device go, those of another device stay
        reset(100, 100);
        ArenaPool a(0), b(0), c(1);
        serve(a, 30);
        serve(b, 40);
        g_hip.device = 1;
        serve(c, 50);
        g_hip.device = 0;
        int *p = nullptr, *q = nullptr;
        const hipError_t e1 = device_malloc(&p, 90), e2 = device_malloc(&q, 90);
        std::printf("pressure %d %d %d %zu %zu %d\n", (int)e1, (int)e2, q == nullptr, 100 - g_hip.room[0],
                    100 - g_hip.room[1], (int)hipGetLastError());
        (void)hipFree(p);
    }
    {
        // a table that cannot grow is gone, not dangling
        reset(100, 0);
        short *t = nullptr;
        size_t cap = 0;
        const hipError_t e1 = device_regrow(t, cap, 20), e2 = device_regrow(t, cap, 21);
        std::printf("table %d %d %zu", (int)e1, (int)e2, cap);
        const hipError_t e3 = device_regrow(t, cap, 60);
        std::printf(" %d %zu %d %zu", (int)e3, cap, t == nullptr, 100 - g_hip.room[0]);
        const hipError_t e4 = device_regrow(t, cap, 10);
        std::printf(" %d %zu %zu\n", (int)e4, cap, 100 - g_hip.room[0]);
    }
    return 0;
}
