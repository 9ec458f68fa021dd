// int8 chains of L = 8, 16, 32 held in the registers of one wave
// (small_core.hpp): Metropolis sweeps (replacing src/ising.cpp:87-149) and the
// measurement of every level (src/lattice.cpp:102-120, src/mcrg.cpp:72-98,
// :314-348).
#include "small_core.hpp"

namespace mcrg {

// One int8 lattice: its words through LDS, n sweeps, all measured or none, and
// its counters.
template <uint32_t L>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void k_small_chain(const HbmLattice *__restrict__ lats, uint32_t n, uint32_t measure)
{
    constexpr uint32_t W = L * L / 64u, half = L / 2u, sites = L * half;
    extern __shared__ uint32_t lds[];
    const HbmLattice &lat = lats[blockIdx.x];
    const uint32_t lane = threadIdx.x, w = lane & (W - 1u);
    // site mc of colour c (checkerboard order) sits at row mc / (L/2)
    auto at = [&](uint32_t mc, uint32_t c) {
        const uint32_t y = mc / half;
        return y * L + 2u * (mc % half) + ((y + c) & 1u);
    };
    for (uint32_t c = 0; c < 2u; ++c)
#pragma unroll
        for (uint32_t m0 = 0; m0 < sites; m0 += 64u) {
            const uint32_t mc = m0 + lane;
            const uint64_t b = __ballot(mc < sites && lat.spins[at(mc & (sites - 1u), c)] < 0);
            if (lane < 2u && (m0 >> 5) + lane < W) lds[c * W + (m0 >> 5) + lane] = (uint32_t)(b >> (32u * lane));
        }
    SmallLattice me{};
    me.alive = true;
    me.k0 = lat.k0;
    me.k1 = lat.k1;
    me.acc = lat.acc;
    me.t = lat.state[0];
    me.therm = measure ? 0u : n;
    me.meas = measure ? n : 0u;
    me.n_measured = lat.state[1];
    me.spb = (uint32_t)lat.sweeps_per_bin;
    me.records = lat.records;
    small_sync();
    uint32_t c0 = lds[w], c1 = lds[W + w];
    small_sync();
    run_small<L>(me, n, (uint32_t)lat.n_levels, 64u, lds, c0, c1);
    small_sync();
    if (lane < W) {
        lds[w] = c0;
        lds[W + w] = c1;
    }
    small_sync();
    for (uint32_t c = 0; c < 2u; ++c)
        for (uint32_t mc = lane; mc < sites; mc += 64u)
            lat.spins[at(mc, c)] = (int8_t)(1 - 2 * (int)((lds[c * W + (mc >> 5)] >> (mc & 31u)) & 1u));
    if (lane == 0u) {
        lat.state[0] = me.t + n;
        lat.state[1] = me.n_measured + me.meas;
    }
}

hipError_t launch_small_chain(const HbmLattice *d, int n_lats, int L, int n_levels, uint32_t n, bool measure,
                              hipStream_t s)
{
    const uint32_t lds_bytes = 4u * small_lds_words((uint32_t)L, 1u, (uint32_t)n_levels);
    const dim3 grid((uint32_t)n_lats), block(64);
    const uint32_t m = measure ? 1u : 0u;
    if (L == 8) hipLaunchKernelGGL(k_small_chain<8u>, grid, block, lds_bytes, s, d, n, m);
    else if (L == 16) hipLaunchKernelGGL(k_small_chain<16u>, grid, block, lds_bytes, s, d, n, m);
    else if (L == 32) hipLaunchKernelGGL(k_small_chain<32u>, grid, block, lds_bytes, s, d, n, m);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace mcrg
