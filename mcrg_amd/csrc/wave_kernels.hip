// Batch and server jobs of 8 <= L <= 128, held in the registers of waves
// (small_core.hpp, wave_core.hpp): Metropolis sweeps (replacing
// src/ising.cpp:87-149) and the measurement of every level
// (src/lattice.cpp:102-120, src/mcrg.cpp:72-98, :314-348).  A slot is one wave:
// one lattice of L = 64 or 128, or 64 / T smaller ones.
//
// One kernel for all sizes, so that a launch of uneven jobs needs one queue and
// every wave is placed at once: with a kernel per size on three streams the
// small lattices' waves ran behind the L = 128 ones (two hardware queues).
#include "wave_core.hpp"

namespace mcrg {

template <uint32_t L>
__device__ __forceinline__ void small_slot(const Slot &sl, const int32_t *__restrict__ slot_lats,
                                           PackedLattice *__restrict__ lats, uint32_t *lds)
{
    constexpr uint32_t W = L * L / 64u;
    const uint32_t T = 64u / (uint32_t)sl.G, lane = threadIdx.x, u = lane & (T - 1u), w = u & (W - 1u);
    const int32_t li = slot_lats[sl.first + (int32_t)(lane / T)];
    SmallLattice me{};
    uint32_t c0 = 0, c1 = 0;
    me.spb = 1u;
    if (li >= 0) {
        const PackedLattice &P = lats[li];
        me.alive = true;
        me.k0 = P.k0;
        me.k1 = P.k1;
        me.acc = P.acc;
        me.t = P.t;
        me.therm = P.therm_left;
        me.meas = P.meas_left;
        me.n_measured = P.n_measured;
        me.spb = (uint32_t)P.sweeps_per_bin;
        me.records = P.records;
        c0 = P.spins[w];
        c1 = P.spins[W + w];
    }
    run_small<L>(me, sl.n_sweeps, (uint32_t)sl.n_levels, T, lds, c0, c1);
    if (li >= 0) {
        PackedLattice &P = lats[li];
        if (u < W) {
            P.spins[w] = c0;
            P.spins[W + w] = c1;
        }
        if (u == 0u) {
            const uint32_t total = me.therm + me.meas, swept = total < sl.n_sweeps ? total : sl.n_sweeps;
            const uint32_t measured = swept > me.therm ? swept - me.therm : 0u;
            P.t = me.t + swept;
            P.n_measured = me.n_measured + measured;
            P.therm_left = me.therm - (swept - measured);
            P.meas_left = me.meas - measured;
        }
    }
}

template <uint32_t L>
__device__ __forceinline__ void wave_slot(const Slot &sl, const int32_t *__restrict__ slot_lats,
                                          PackedLattice *__restrict__ lats, uint32_t *lds)
{
    constexpr uint32_t WPL = WaveGeom<L>::WPL, W = L * L / 64u;
    const int32_t li = slot_lats[sl.first];
    if (li < 0) return;
    const uint32_t lane = threadIdx.x;
    PackedLattice &P = lats[li];
    SmallLattice me;
    me.alive = true;
    me.k0 = P.k0;
    me.k1 = P.k1;
    me.acc = P.acc;
    me.t = P.t;
    me.therm = P.therm_left;
    me.meas = P.meas_left;
    me.n_measured = P.n_measured;
    me.spb = (uint32_t)P.sweeps_per_bin;
    me.records = P.records;
    uint32_t c0[WPL], c1[WPL];
#pragma unroll
    for (uint32_t k = 0; k < WPL; ++k) {
        c0[k] = P.spins[WPL * lane + k];
        c1[k] = P.spins[W + WPL * lane + k];
    }
    run_wave<L>(me, sl.n_sweeps, (uint32_t)sl.n_levels, lds, c0, c1);
#pragma unroll
    for (uint32_t k = 0; k < WPL; ++k) {
        P.spins[WPL * lane + k] = c0[k];
        P.spins[W + WPL * lane + k] = c1[k];
    }
    if (lane == 0u) {
        const uint32_t total = me.therm + me.meas, swept = total < sl.n_sweeps ? total : sl.n_sweeps;
        const uint32_t measured = swept > me.therm ? swept - me.therm : 0u;
        P.t = me.t + swept;
        P.n_measured = me.n_measured + measured;
        P.therm_left = me.therm - (swept - measured);
        P.meas_left = me.meas - measured;
    }
}

__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void k_wave(
    const Slot *__restrict__ slots, const int32_t *__restrict__ slot_lats, PackedLattice *__restrict__ lats)
{
    extern __shared__ uint32_t lds[];
    const Slot sl = slots[blockIdx.x];
    switch (sl.L) {
    case 8: small_slot<8u>(sl, slot_lats, lats, lds); break;
    case 16: small_slot<16u>(sl, slot_lats, lats, lds); break;
    case 32: small_slot<32u>(sl, slot_lats, lats, lds); break;
    case 64: wave_slot<64u>(sl, slot_lats, lats, lds); break;
    default: wave_slot<128u>(sl, slot_lats, lats, lds); break;
    }
}

hipError_t launch_wave(const Slot *slots, uint32_t n_slots, const int32_t *slot_lats, PackedLattice *lats,
                       uint32_t lds_bytes, hipStream_t s)
{
    hipLaunchKernelGGL(k_wave, dim3(n_slots), dim3(64), lds_bytes, s, slots, slot_lats, lats);
    return hipGetLastError();
}

}  // namespace mcrg
