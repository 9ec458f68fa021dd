// Resident schedule: bit-packed (CB) lattices held in a wave's registers (L <=
// 128) or a workgroup's LDS (L = 256, 512) for a whole chunk of sweeps.  A
// "slot" is G lattices of one side L and one level count that a wave advances
// together, or one lattice of a workgroup; a persistent grid of workgroups
// pulls those from a queue.  Shared by the host engine and the kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_common.hpp"
#include "hbm_kernels.hpp"

namespace mcrg {

constexpr int kResidentMinL = 8;
constexpr int kResidentMaxL = 512;
constexpr uint32_t kMetaWords = 16;
constexpr uint32_t kMaxLdsBytes = 160u * 1024u - 64u;

// Per-lattice (job) state in device memory.
struct PackedLattice {
    uint32_t *spins;      // CB words: colour 0 [W] then colour 1 [W], W = L*L/64
    int64_t *records;     // max_bins * record_size(n_levels)
    uint32_t k0, k1;      // Philox key = seed
    Accept acc;
    uint32_t t;           // next sweep index
    uint32_t n_measured;  // measured samples so far
    uint32_t therm_left;  // unmeasured sweeps still to run
    uint32_t meas_left;   // measured sweeps still to run
    int32_t L, n_levels, sweeps_per_bin, max_bins;
};

// G lattice positions of one (L, n_levels) class: slot_lats[first .. first+G),
// -1 marks an empty position.
struct Slot {
    int32_t L, G, n_levels, first;
    uint32_t n_sweeps;  // sweeps this launch advances each lattice of the slot (at most)
};

__host__ __device__ inline uint32_t cb_words(uint32_t L) { return L * L / 64u; }

__host__ __device__ inline uint32_t level_words(uint32_t L, uint32_t l)
{
    const uint32_t Ll = L >> l;
    const uint32_t w = (Ll * Ll + 31u) / 32u;
    return w ? w : 1u;
}

// LDS words that a server's admission counts for G lattices of a workgroup, T =
// threads per lattice: spins, blocked levels and their tie coins, counts,
// operator values and records.  A weight by which the budget limits the resident
// jobs (and refuses some), not what a launch takes: big_layout() (1.1 k to 3.3 k
// words more for a lattice, since 64 samples wait there), wave_lds_words() (half
// a thousand words more for L = 64, a hundred to two hundred less for L = 128 with
// two levels or more) or small_lds_words().
__host__ __device__ inline uint32_t slot_words(uint32_t L, uint32_t G, uint32_t nl, uint32_t T)
{
    uint32_t lvl = 0;
    for (uint32_t l = 1; l <= nl; ++l) lvl += level_words(L, l);
    const uint32_t counts = (T > 64u ? T / 64u : 1u) * (nl + 1u) * 4u, values = 3u * (nl + 1u) + 3u;
    const uint32_t before = G * (kMetaWords + 2u * cb_words(L) + 2u * lvl + counts + values) + record_size(nl);
    return ((before + 1u) & ~1u) + G * record_size(nl) * 2u;
}

// Admits n lattices: lats[idx[k]] = stage[k], its records zeroed, its spins
// drawn (stage and idx in device memory).
hipError_t launch_packed_init(PackedLattice *lats, const PackedLattice *stage, const int32_t *idx, int n,
                              hipStream_t s);
// Work items of one launch: sub-chunk k (0 <= k < n_sub) of slot i is item
// k * n_slots + i, so that every slot's first part is queued before any second
// part.  Sub-chunk k runs sweeps [k c, min((k+1) c, n_sweeps)) of its slot,
// c = ceil(n_sweeps / n_sub), and starts only after sub-chunk k-1 of the same
// slot has published its write-back (done[i] = k); with n_sub = 1 there is no
// waiting.  `done` holds n_slots words and `queue` one, both zeroed by the
// launch; a wait that exceeds kSubChunkWaitTicks sets *err.
constexpr uint64_t kSubChunkWaitTicks = 2000000000ull;  // 20 s of the 100 MHz clock
hipError_t launch_resident(int threads, const Slot *slots, uint32_t n_slots, uint32_t n_sub,
                           const int32_t *slot_lats, PackedLattice *lats, uint32_t *queue, uint32_t *done,
                           uint32_t *err, uint32_t lds_bytes, uint32_t grid, hipStream_t s);
int resident_max_active_groups(int threads, uint32_t lds_bytes);
// Slots of one wave each: one lattice of L = 64 or 128 (wave_core.hpp), or G
// smaller ones, G a power of two, at most 64 / cb_words(L) (small_core.hpp).
constexpr int kSmallMaxL = 32, kWaveMaxL = 128;
hipError_t launch_wave(const Slot *slots, uint32_t n_slots, const int32_t *slot_lats, PackedLattice *lats,
                       uint32_t lds_bytes, hipStream_t s);

}  // namespace mcrg
