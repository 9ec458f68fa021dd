// int8 chains of L = 64 and 128 in one workgroup, its waves split by colour:
// Metropolis sweeps (replacing src/ising.cpp:87-149) and the measurement of
// every level (src/lattice.cpp:102-120, src/mcrg.cpp:72-98, :314-348).
#include <algorithm>
#include <cstdlib>

#include "lds_opt_in.hpp"
#include "wave_core.hpp"

namespace mcrg {

// SETS sets of W / 64 waves, a word a lane, take the half sweeps in turn: a set
// draws its next random numbers while the others decide, so that a half sweep
// lasts as long as its reads, its decisions and its stores.  A sweep's words go
// to one of kRing buffers in LDS, each with the number of its sweep, in one
// 64-bit store: whoever reads words polls them until they are the sweep's, so
// there is neither a barrier nor a flag between a word and the decisions that
// wait for it.  The last M waves take the samples in turn (wave_core.hpp's two
// steps) and hold nobody up until they are a ring behind.
//
// Why every wait ends: a word is waited for only by the work that comes after it
// in the order colour 0, colour 1, sample of each sweep, and a sample by colour
// 0 kRing sweeps later; every wave goes through its steps in that order, and all
// waves of a workgroup are resident.  Why no word is overwritten too early: a
// word of sweep t is stored after its neighbours' and its own of half a sweep
// and a sweep before have been read, whose lanes had by then read everything up
// to sweep t - 1, and colour 0 waits for the sample of sweep t - kRing.  Polls
// are counted all the same: a wave that gives up ends with the step it is in, the
// others, who wait for its words, do so as well, and the error word says that the
// state is lost (leaving the step at once took L = 128 6 % more time: its branch
// stands between the words and their decisions).  The count costs a poll 6 % of a
// half sweep at L = 64; one comparison of everything that is waited for, instead
// of one a word and their masks joined, gives that back and more.
//
// Bound by the latency of a half sweep (L = 64: 720 cycles) and, at L = 128, by
// VALU issue (8 wave-words a sweep on each SIMD).  us a sweep, unmeasured and
// measured, against strips on many compute units: L = 64 2.41 -> 0.60 and 3.01 ->
// 0.70; L = 128 2.40 -> 1.04 and 2.64 -> 1.14.  One lattice: two sets take 0.70
// and 0.78 at L = 64, three sets 1.02 and 1.34 at L = 128 (four measuring waves;
// two 1.91); with the random numbers drawn when the words are there L = 64 takes
// 1.09, with one refinement call ahead instead of two 0.85.  Groups of lattices:
// 256 x L = 64 8.1 -> 0.7 and 20.7 -> 1.0, 4096 x L = 128 70 -> 18 and 137 -> 22.
template <uint32_t L>
struct ColourGeom {
    static constexpr uint32_t W = L * L / 64u, NW = W / 64u;
    static constexpr uint32_t SETS = L == 64u ? 4u : 2u, M = L == 64u ? 4u : 8u;
    static constexpr uint32_t waves = SETS * NW + M, threads = 64u * waves;
    static constexpr uint32_t entry = WaveGeom<L>::stride;
};
constexpr uint32_t kRing = 8u;

template <uint32_t L>
static uint32_t colour_lds_words(uint32_t nl)
{
    using G = ColourGeom<L>;
    return kRing * 4u * G::W + G::M + 2u + G::M * 64u * G::entry + 2u * G::M * record_size(nl);
}

__device__ __forceinline__ uint64_t word_ld(const uint64_t *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// One lattice: n sweeps, all measured or none, and its counters.
template <uint32_t L>
__global__ __launch_bounds__(ColourGeom<L>::threads) void k_colour_chain(const HbmLattice *__restrict__ lats, uint32_t n,
                                                                         uint32_t measure, uint32_t spins)
{
    using G = ColourGeom<L>;
    constexpr uint32_t W = G::W, NW = G::NW, M = G::M, half = L / 2u, sites = L * half, WPR = L / 64u;
    static_assert(kRing % M == 0u, "the sample that a buffer holds");
    extern __shared__ __align__(16) uint32_t lds[];
    uint64_t *ring = reinterpret_cast<uint64_t *>(lds);  // word | sweeps done << 32
    uint32_t *read = lds + kRing * 4u * W, *lost = read + M, *samples = lost + 2;  // lost: 1 once a wave gave up
    const HbmLattice &lat = lats[blockIdx.x];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = uni<true>(tid >> 6);
    const uint32_t nl = (uint32_t)lat.n_levels, rs = record_size(nl), t0 = lat.state[0], q0 = lat.state[1];
    // site mc of colour c (checkerboard order) sits at row mc / (L/2)
    auto at = [&](uint32_t mc, uint32_t c) {
        const uint32_t y = mc / half;
        return y * L + 2u * (mc % half) + ((y + c) & 1u);
    };
    for (uint32_t k = tid; k < kRing * 2u * W; k += G::threads)
        if (k >= 2u * W) ring[k] = 0u;
    if (tid <= M) read[tid] = 0u;
    for (uint32_t m0 = 64u * wave; m0 < 2u * sites; m0 += G::threads) {
        const uint32_t c = m0 >= sites ? 1u : 0u, mc = m0 - c * sites + lane;
        const uint64_t b = __ballot(lat.spins[at(mc, c)] < 0);
        if (lane < 2u) ring[(m0 >> 5) + lane] = (uint32_t)(b >> (32u * lane));
    }
    __syncthreads();
    const uint32_t k0 = lat.k0, k1 = lat.k1;
    if (wave < G::SETS * NW) {
        __builtin_amdgcn_s_setprio(3);
        const uint32_t set = wave / NW, word = 64u * (wave - set * NW) + lane, y = word / WPR, q = word % WPR;
        const uint32_t up = ((y - 1u) & (L - 1u)) * WPR + q, dn = ((y + 1u) & (L - 1u)) * WPR + q;
        const Accept acc = lat.acc;
        uint32_t end = 2u * n;
        for (uint32_t step = set; step < end; step += G::SETS) {
            const uint32_t it = step >> 1, c = step & 1u, t = t0 + it, have = it + c, p = (y + c) & 1u;
            const MetropolisAhead<2u> h = metropolis_ahead<2u>(acc, k0, k1, word, t, c);
            const uint64_t *mine = ring + (it % kRing) * 2u * W + c * W;
            const uint64_t *oth = ring + (have % kRing) * 2u * W + (1u - c) * W;
            const uint32_t beside = y * WPR + ((q + 2u * p - 1u) & (WPR - 1u));
            // colour 0 writes over the sample of kRing sweeps ago
            const uint32_t want = c == 0u && measure && it >= kRing ? it - kRing + 1u : 0u;
            uint64_t own, o, side, nu, nd;
            uint32_t left = spins;
            for (;;) {
                const uint32_t done = want ? lds_ld(read + (it % M)) : 0u;
                own = word_ld(mine + word);
                o = word_ld(oth + word);
                side = WPR == 1u ? o : word_ld(oth + beside);
                nu = word_ld(oth + up);
                nd = word_ld(oth + dn);
                uint32_t off = ((uint32_t)(own >> 32) ^ it) | ((uint32_t)(o >> 32) ^ have) |
                               ((uint32_t)(side >> 32) ^ have) | ((uint32_t)(nu >> 32) ^ have) |
                               ((uint32_t)(nd >> 32) ^ have);
                off |= done < want ? 1u : 0u;
                asm("" : "+v"(off));  // one comparison, not one a word and their masks joined
                if (__builtin_amdgcn_ballot_w64(off != 0u) == 0ull) break;
                if (left-- == 0u) {  // the last step, from whatever is there
                    lds_st(lost, 1u);
                    end = 0u;
                    break;
                }
            }
            const uint32_t w = (uint32_t)own ^
                               metropolis_decide(h, (uint32_t)own, (uint32_t)nu, (uint32_t)nd,
                                                 row_left((uint32_t)o, (uint32_t)side, p != 0u),
                                                 row_right((uint32_t)o, (uint32_t)side, p != 0u), acc, k0, k1, word, t, c);
            __hip_atomic_store(ring + ((it + 1u) % kRing) * 2u * W + c * W + word, (uint64_t)w | ((uint64_t)(it + 1u) << 32),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    } else if (measure) {
        const uint32_t j = wave - G::SETS * NW;
        uint32_t *mine = samples + j * 64u * G::entry;
        int64_t *rec = reinterpret_cast<int64_t *>(samples + M * 64u * G::entry) + j * rs;
        for (uint32_t k = lane; k < rs; k += 64u) rec[k] = 0;
        uint32_t rec_bin = 0xFFFFFFFFu, slot = 0, end = n;
        auto flush = [&]() {
            small_sync();
            // the measuring waves share bins
            for (uint32_t k = lane; k < rs; k += 64u)
                __hip_atomic_fetch_add(reinterpret_cast<unsigned long long *>(lat.records) + (size_t)rec_bin * rs + k,
                                       (unsigned long long)rec[record_canon(nl, k)], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
            small_sync();
            for (uint32_t k = lane; k < rs; k += 64u) rec[k] = 0;
            small_sync();
        };
        for (uint32_t it = j; it < end; it += M) {
            constexpr uint32_t WPL = WaveGeom<L>::WPL;
            const uint64_t *buf = ring + ((it + 1u) % kRing) * 2u * W + WPL * lane;
            uint32_t c0[WPL], c1[WPL];
            for (uint32_t left = spins;; --left) {
                uint32_t off = 0;
#pragma unroll
                for (uint32_t k = 0; k < WPL; ++k) {
                    const uint64_t a = word_ld(buf + k), b = word_ld(buf + W + k);
                    c0[k] = (uint32_t)a;
                    c1[k] = (uint32_t)b;
                    off |= ((uint32_t)(a >> 32) ^ (it + 1u)) | ((uint32_t)(b >> 32) ^ (it + 1u));
                }
                if (__builtin_amdgcn_ballot_w64(off != 0u) == 0ull) break;
                if (left == 0u) {
                    lds_st(lost, 1u);
                    end = 0u;
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
            if (lane == 0u) lds_st(read + j, it + 1u);
            wave_sample<L>(c0, c1, nl, t0 + it, k0, k1, mine + slot * G::entry);
            ++slot;
            if (slot < 64u && it + M < n) continue;
            // lane u finishes the u-th of the last `slot` samples
            small_sync();
            const uint32_t first = it - (slot - 1u) * M, i = first + lane * M;
            wave_finish<L>(mine + lane * G::entry, nl, k0, k1, t0 + i, (q0 + i) / (uint32_t)lat.sweeps_per_bin,
                           lane < slot, rec, rec_bin, flush);
            slot = 0;
            small_sync();
        }
        if (rec_bin != 0xFFFFFFFFu) flush();
    }
    __syncthreads();
    if (lds_ld(lost) != 0u) {
        if (tid == 0u) __hip_atomic_store(lat.error, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        return;
    }
    const uint64_t *end = ring + (n % kRing) * 2u * W;
    for (uint32_t mc = tid; mc < 2u * sites; mc += G::threads) {
        const uint32_t c = mc >= sites ? 1u : 0u;
        lat.spins[at(mc - c * sites, c)] = (int8_t)(1 - 2 * (int)(((uint32_t)end[mc >> 5] >> (mc & 31u)) & 1u));
    }
    if (tid == 0u) {
        lat.state[0] = t0 + n;
        lat.state[1] = q0 + (measure ? n : 0u);
    }
}

template <uint32_t L>
static hipError_t launch_colour(const HbmLattice *d, int n_lats, int n_levels, uint32_t n, bool measure, hipStream_t s)
{
    const uint32_t lds_bytes = 4u * colour_lds_words<L>((uint32_t)n_levels);  // L = 128: up to 72,992 bytes
    static LdsOptIn lds;
    const hipError_t le = lds.need(reinterpret_cast<const void *>(&k_colour_chain<L>), lds_bytes);
    if (le != hipSuccess) return le;
    uint32_t spins = kColourSpins;
    if (const char *v = std::getenv("MCRG_COLOUR_SPINS")) spins = (uint32_t)std::min<long>(std::max(0L, std::atol(v)), kColourSpins);
    hipLaunchKernelGGL(k_colour_chain<L>, dim3((uint32_t)n_lats), dim3(ColourGeom<L>::threads), lds_bytes, s, d, n,
                       measure ? 1u : 0u, spins);
    return hipGetLastError();
}

hipError_t launch_colour_chain(const HbmLattice *d, int n_lats, int L, int n_levels, uint32_t n, bool measure,
                               hipStream_t s)
{
    if (L == 64) return launch_colour<64u>(d, n_lats, n_levels, n, measure, s);
    if (L == 128) return launch_colour<128u>(d, n_lats, n_levels, n, measure, s);
    return hipErrorInvalidValue;
}

}  // namespace mcrg
