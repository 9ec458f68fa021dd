// LdsOptIn (csrc/lds_opt_in.hpp) on the stand-in devices of tests/cpp/fake_hip:
// for each call the device, the bytes, the result, the kernel's level there and
// the attribute calls so far, for tests/test_lds_opt_in_cpu.py.
#include <cstdio>

#include "../../mcrg_amd/csrc/lds_opt_in.hpp"

int main()
{
    mcrg::LdsOptIn lds;
    const int kernel = 0;
    g_hip.set_max = 160 * 1024;
    const int calls[][2] = {{0, 65536}, {0, 70000}, {0, 66000}, {1, 66000}, {1, 90000}, {0, 80000},
                            {1, 80000}, {0, 200000}, {0, 80000}, {0, 100000}};
    for (auto &c : calls) {
        g_hip.device = c[0];
        const hipError_t e = lds.need(&kernel, (uint32_t)c[1]);
        std::printf("%d %d %d %d %d\n", c[0], c[1], (int)e, g_hip.lds[{c[0], &kernel}], g_hip.set_calls);
    }
    return 0;
}
