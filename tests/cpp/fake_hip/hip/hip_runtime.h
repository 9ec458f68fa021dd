// A stand-in for the HIP runtime's memory and attribute calls: devices of a few
// bytes each, in host memory, for tests of the code that allocates and launches
// (no GPU).
#pragma once
#include <cstddef>
#include <cstdlib>
#include <map>
#include <utility>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };

struct FakeHip {
    size_t room[2] = {0, 0};
    int device = 0, frees = 0;
    hipError_t last = hipSuccess;
    std::map<void *, std::pair<int, size_t>> live;
    int set_calls = 0, set_max = 1 << 30;
    std::map<std::pair<int, const void *>, int> lds;  // (device, kernel) -> dynamic LDS it may take
};
inline FakeHip g_hip;

inline hipError_t hipGetDevice(int *d)
{
    *d = g_hip.device;
    return hipSuccess;
}
inline hipError_t hipMalloc(void **p, size_t bytes)
{
    if (bytes > g_hip.room[g_hip.device]) return g_hip.last = hipErrorOutOfMemory;
    g_hip.room[g_hip.device] -= bytes;
    *p = std::malloc(1);
    g_hip.live[*p] = {g_hip.device, bytes};
    return hipSuccess;
}
inline hipError_t hipFree(void *p)
{
    auto it = g_hip.live.find(p);
    if (it == g_hip.live.end()) return g_hip.last = hipErrorInvalidValue;
    g_hip.room[it->second.first] += it->second.second;
    g_hip.live.erase(it);
    std::free(p);
    ++g_hip.frees;
    return hipSuccess;
}
inline hipError_t hipGetLastError()
{
    const hipError_t e = g_hip.last;
    g_hip.last = hipSuccess;
    return e;
}

enum hipFuncAttribute { hipFuncAttributeMaxDynamicSharedMemorySize = 8 };
inline hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute, int value)
{
    ++g_hip.set_calls;
    if (value > g_hip.set_max) return hipErrorInvalidValue;
    g_hip.lds[{g_hip.device, f}] = value;
    return hipSuccess;
}
