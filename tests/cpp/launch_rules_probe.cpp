// Host-side launch rules on their own, for tests/test_launch_rules_cpu.py: reads
// "sw_lds need n_lats n_cus" lines and prints the bytes a workgroup asks for.
#include <cstdio>
#include <cstring>

#include "../../mcrg_amd/csrc/hbm_kernels.hpp"

int main()
{
    char what[32];
    unsigned need;
    int n_lats, n_cus;
    while (std::scanf("%31s %u %d %d", what, &need, &n_lats, &n_cus) == 4)
        if (std::strcmp(what, "sw_lds") == 0) std::printf("%u\n", mcrg::sw_wg_lds_bytes(need, n_lats, n_cus));
    return 0;
}
