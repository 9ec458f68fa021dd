// Small lattices (L = 8, 16, 32) in the registers of one wave.
//
// A lattice of W = L^2/64 words per colour has a team of T lanes (W <= T <= 64,
// a power of two), a wave 64 / T lattices.  Lane u of a team holds word
// w = u mod W of both colours; the T / W groups of W lanes hold copies and do
// the same updates.  Neighbour words come from DPP rotations within a group, so
// a sweep touches neither LDS nor a barrier.  What the copies are for:
//   * group j draws and prepares the random numbers of sweep it0 + j, both
//     colours, and every group fetches them a sweep before they are due: one draw per
//     T / W sweeps;
//   * samples are kept in LDS as words, and once T sweeps have passed lane u
//     measures sample u by itself, whole levels as words in registers: no lane
//     idles and nothing is reduced but the record's terms.
// Bound by the latency of a wave's dependent instructions (a measured sweep of
// one lattice 0.52 us at L = 8, 0.64 at 16, 0.95 at 32, unmeasured 0.41, 0.47 and
// 0.68; with the numbers fetched in the sweep that needs them 0.56, 0.72 and 0.98,
// and with the calls' words as they are drawn 0.73, 0.89 and 1.11); teams of 4 or 16 lanes in
// a workgroup's LDS took 8 to 10 us, and one launch per phase 32 us.
#pragma once

#include "levels.hpp"
#include "resident.hpp"
#include "resident_core.hpp"

namespace mcrg {

// LDS of one wave, in 32-bit words: the samples of a block (an odd stride, so
// that the lanes' words lie in different banks), then per lattice the partial
// record of the bin in progress.
__host__ __device__ inline uint32_t small_snap_stride(uint32_t L) { return 2u * cb_words(L) + 1u; }
__host__ __device__ inline uint32_t small_lds_words(uint32_t L, uint32_t G, uint32_t nl)
{
    return ((64u * small_snap_stride(L) + 1u) & ~1u) + 2u * G * record_size(nl);
}

// Value of the next (previous) lane of the aligned group of W lanes.
template <uint32_t W>
__device__ __forceinline__ uint32_t lane_next(uint32_t v)
{
    if (W == 4u) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x39, 0xF, 0xF, false);    // quad_perm 1,2,3,0
    if (W == 16u) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x12F, 0xF, 0xF, false);  // row_ror:15
    return v;
}
template <uint32_t W>
__device__ __forceinline__ uint32_t lane_prev(uint32_t v)
{
    if (W == 4u) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x93, 0xF, 0xF, false);    // quad_perm 3,0,1,2
    if (W == 16u) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x121, 0xF, 0xF, false);  // row_ror:1
    return v;
}

// What a lane knows of its lattice.
struct SmallLattice {
    bool alive;
    uint32_t k0, k1;
    Accept acc;
    uint32_t t, therm, meas;       // next sweep, unmeasured and measured sweeps left
    uint32_t n_measured, spb;      // samples before, samples per bin
    int64_t *records;
};

// ------------------------------------------------------------------ measurement
// Operator counts of a row-major level of side Ll (whole, N words of which the
// last may be short): disagreements NN, NNN, P.
template <uint32_t Ll>
struct SmallLevel {
    static constexpr uint32_t n = Ll * Ll;
    static constexpr uint32_t N = (n + 31u) / 32u;
    uint32_t w[N];

    // bit b: the site right of (below) bit b of word i
    static __device__ __forceinline__ uint32_t right(uint32_t v)
    {
        constexpr uint32_t e = Ll == 16u ? 0x80008000u : Ll == 8u ? 0x80808080u : Ll == 4u ? 0x88888888u : 0xAAAAAAAAu;
        return ((v >> 1) & ~e) | ((v << (Ll - 1u)) & e);
    }
    __device__ __forceinline__ uint32_t down(uint32_t i) const
    {
        if (n >= 32u) return (w[i] >> Ll) | (w[(i + 1u) % N] << (32u - Ll));
        return ((w[0] >> Ll) | (w[0] << (n - Ll))) & ((1u << (n & 31u)) - 1u);
    }
    __device__ __forceinline__ void ops(int32_t S[3]) const
    {
        uint32_t dnn = 0, dnnn = 0, dp = 0;
        constexpr uint32_t valid = n >= 32u ? 0xFFFFFFFFu : (1u << (n & 31u)) - 1u;
#pragma unroll
        for (uint32_t i = 0; i < N; ++i) {
            const uint32_t a = w[i], d = down(i), r = right(a) & valid, g = right(d) & valid;
            dnn += (uint32_t)(popc(a ^ r) + popc(a ^ d));
            dnnn += (uint32_t)(popc(a ^ g) + popc(r ^ d));
            dp += (uint32_t)popc(xor3(a, r, d) ^ g);
        }
        S[0] = (int32_t)(2u * n) - 2 * (int32_t)dnn;
        S[1] = (int32_t)(2u * n) - 2 * (int32_t)dnnn;
        S[2] = (int32_t)n - 2 * (int32_t)dp;
    }
    // b = 2 majority blocking, ties take the bits of coin (the stream's words
    // for the blocked level).
    __device__ __forceinline__ SmallLevel<Ll / 2u> block(const uint32_t coin[4]) const
    {
        constexpr uint32_t Lb = Ll / 2u, pairs = 32u / (2u * Ll) ? 32u / (2u * Ll) : 1u;  // row pairs of a word
        SmallLevel<Lb> o;
#pragma unroll
        for (uint32_t k = 0; k < SmallLevel<Lb>::N; ++k) o.w[k] = 0;
#pragma unroll
        for (uint32_t by = 0; by < Lb; ++by) {
            const uint32_t i = by / pairs, sh = by % pairs * 2u * Ll;
            const uint32_t r0 = w[i] >> sh, r1 = w[i] >> (sh + Ll), at = by * Lb;
            const uint32_t bits = block16(r0, r1, coin[at >> 5] >> (at & 31u)) & ((1u << Lb) - 1u);
            o.w[at >> 5] |= bits << (at & 31u);
        }
        return o;
    }
};

// Operators of the levels from l on (x is level l, side Ll) into S[l..nl].
// draw(call, level, out) gives four words of the level's tie coins.
template <uint32_t Ll, uint32_t l, uint32_t NLMAX, typename Draw>
__device__ __forceinline__ void small_levels(const SmallLevel<Ll> &x, uint32_t nl, int32_t (&S)[NLMAX + 1u][3], Draw draw)
{
    if (l > nl) return;
    x.ops(S[l]);
    if constexpr (Ll > 2u) {
        if (l < nl) {
            uint32_t coin[4];
            draw(0u, l, coin);
            small_levels<Ll / 2u, l + 1u, NLMAX>(x.block(coin), nl, S, draw);
        }
    }
}

// Level 0 of one sample (its checkerboard words at snap: colour 0, then colour
// 1) and the blocking into level 1.
template <uint32_t L>
__device__ __forceinline__ SmallLevel<L / 2u> small_level0(const uint32_t *snap, const uint32_t *coin, int32_t S[3],
                                                           int32_t &M)
{
    constexpr uint32_t W = L * L / 64u, Lb = L / 2u;
    const uint32_t *c0 = snap, *c1 = snap + W;
    uint32_t dnn = 0, dnnn = 0, dp = 0, nd = 0;
    // two words at a time: unrolled whole, L = 32 took 248 VGPRs, and its waves
    // share the SIMDs with the other lattices'
#pragma unroll 2
    for (uint32_t w = 0; w < W; ++w) {
        cb_ops_item(c0, c1, L, W, w, 0u, dnn, dnnn, dp, nd);
        cb_ops_item(c1, c0, L, W, w, 1u, dnn, dnnn, dp, nd);
    }
    constexpr int32_t n = (int32_t)(L * L);
    S[0] = 2 * n - 2 * (int32_t)dnn;
    S[1] = 2 * n - 2 * (int32_t)dnnn;
    S[2] = n - 2 * (int32_t)dp;
    M = n - 2 * (int32_t)nd;
    SmallLevel<Lb> o;
#pragma unroll
    for (uint32_t i = 0; i < SmallLevel<Lb>::N; ++i) o.w[i] = cb_block_item(c0, c1, L, W, i, coin[i]);
    return o;
}

__device__ __forceinline__ void small_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Sum over the aligned group of T lanes, in every lane of it below its middle.
__device__ __forceinline__ int32_t team_sum(int32_t v, uint32_t T) { return (int32_t)group_sum((uint32_t)v, T); }

// The partial record of a team's lattice: entries whose two operators are
// exchanged stand once (those with a <= b).
__device__ __forceinline__ uint32_t record_canon(uint32_t nl, uint32_t k)
{
    const uint32_t n_s = 3u * (nl + 1u);
    if (k < n_s || k >= n_s + 9u * (nl + 1u)) return k;
    const uint32_t kk = k - n_s, l = kk / 9u, r = kk % 9u, a = r % 3u, b = r / 3u;
    return a <= b ? k : n_s + 9u * l + 3u * a + b;
}

// Adds the block's samples with `take` to the partial record: every term is
// summed over the team and added by its first lane.  |terms| <= 2^22 for
// L <= 32, so sums over 64 samples fit 32 bits.
template <uint32_t NLMAX>
__device__ __forceinline__ void small_accumulate(int64_t *rec, const int32_t (&S)[NLMAX + 1u][3], int32_t M, bool take,
                                                 uint32_t nl, uint32_t T, bool first_lane)
{
    const uint32_t self = 3u * (nl + 1u), cross = 12u * (nl + 1u), nn0 = cross + 9u * nl, tail = nn0 + nl;
    auto sum = [&](int32_t v) { return team_sum(take ? v : 0, T); };
    auto add = [&](uint32_t k, int32_t v) {
        __hip_atomic_fetch_add(reinterpret_cast<unsigned long long *>(rec + k), (unsigned long long)(int64_t)v,
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
#pragma unroll
    for (uint32_t l = 0; l <= NLMAX; ++l) {
        if (l > nl) break;
#pragma unroll
        for (uint32_t b = 0; b < 3u; ++b) {
            const int32_t sb = sum(S[l][b]);
            int32_t p[3] = {0, 0, 0}, c[3] = {0, 0, 0};
#pragma unroll
            for (uint32_t a = 0; a <= b; ++a) p[a] = sum(S[l][a] * S[l][b]);
            if (l > 0u) {
#pragma unroll
                for (uint32_t a = 0; a < 3u; ++a) c[a] = sum(S[l][a] * S[l - (l > 0u)][b]);
            }
            if (first_lane) {
                add(3u * l + b, sb);
#pragma unroll
                for (uint32_t a = 0; a <= b; ++a) add(self + 9u * l + 3u * b + a, p[a]);
                if (l > 0u) {
#pragma unroll
                    for (uint32_t a = 0; a < 3u; ++a) add(cross + 9u * (l - 1u) + 3u * b + a, c[a]);
                }
            }
        }
        if (l > 0u) {
            const int32_t z = sum(S[l][0] * S[0][0]);
            if (first_lane) add(nn0 + l - 1u, z);
        }
    }
    const int32_t m = sum(M), ma = sum(M < 0 ? -M : M), mm = sum(M * M), one = sum(1);
    if (first_lane) {
        add(tail, m);
        add(tail + 1u, ma);
        add(tail + 2u, mm);
        add(tail + 3u, one);
    }
}

// A word's random numbers as metropolis_ahead prepares them, the outcomes of its
// four ranks as bits (class 1 from bit 0, class 2 from bit 4): a lane prepares one
// sweep of a team's B at a time, and five words a half sweep go to the lanes that
// decide, which then have 65 instructions instead of 95 and eight words.
struct SmallDraw {
    uint32_t a1, o1, a2, o2, ranks;
};

__device__ __forceinline__ SmallDraw small_draw(const Accept &acc, uint32_t k0, uint32_t k1, uint32_t word, uint32_t t,
                                                uint32_t colour)
{
    const MetropolisAhead<1u> h = metropolis_ahead<1u>(acc, k0, k1, word, t, colour);
    uint32_t ranks = 0;
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) ranks |= (h.p1[k] & (1u << k)) | (h.p2[k] & (16u << k));
    return SmallDraw{h.a1, h.o1, h.a2, h.o2, ranks};
}

__device__ __forceinline__ uint32_t small_decide(const SmallDraw &d, uint32_t s, const Nbr4 &nb, const Accept &acc,
                                                 uint32_t k0, uint32_t k1, uint32_t word, uint32_t t, uint32_t colour)
{
    MetropolisAhead<1u> h;
    h.a1 = d.a1;
    h.o1 = d.o1;
    h.a2 = d.a2;
    h.o2 = d.o2;
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) {
        h.p1[k] = (uint32_t)((int32_t)(d.ranks << (31u - k)) >> 31);
        h.p2[k] = (uint32_t)((int32_t)(d.ranks << (27u - k)) >> 31);
    }
    return metropolis_decide<1u>(h, s, nb.nu, nb.nd, nb.nl, nb.nr, acc, k0, k1, word, t, colour);
}

// ------------------------------------------------------------------ the run
// Advances the wave's lattices by up to n sweeps.  c0, c1 are the lane's words;
// nl blockings; `lds` small_lds_words(L, 64 / T, nl) words.
template <uint32_t L>
__device__ __forceinline__ void run_small(const SmallLattice &me, uint32_t n, uint32_t nl, uint32_t T, uint32_t *lds, uint32_t &c0,
                          uint32_t &c1)
{
    constexpr uint32_t W = L * L / 64u, NLMAX = L == 8u ? 2u : L == 16u ? 3u : 4u;
    const uint32_t lane = threadIdx.x & 63u, u = lane & (T - 1u), w = u & (W - 1u), B = T / W, g = lane / T;
    const uint32_t stride = small_snap_stride(L), rs = record_size(nl);
    uint32_t *snap = lds + g * T * stride;
    int64_t *rec = reinterpret_cast<int64_t *>(lds + ((64u * stride + 1u) & ~1u)) + g * rs;
    const uint32_t total = me.alive ? me.therm + me.meas : 0u;
    for (uint32_t k = u; k < rs; k += T) rec[k] = 0;
    uint32_t rec_bin = 0xFFFFFFFFu;  // the bin that rec holds
    const uint64_t team = T == 64u ? ~0ull : ((1ull << T) - 1ull) << (g * T);
    auto flush = [&](bool due) {
        small_sync();
        if (due)
            for (uint32_t k = u; k < rs; k += T) me.records[(size_t)rec_bin * rs + k] += rec[record_canon(nl, k)];
        small_sync();
        if (due)
            for (uint32_t k = u; k < rs; k += T) rec[k] = 0;
        small_sync();
    };
    // the longest run and the first sample of any lattice of the wave
    uint32_t last = total < n ? total : n, begin = me.alive && me.meas > 0u ? me.therm : 0xFFFFFFFFu;
    for (uint32_t o = 32u; o >= 1u; o >>= 1) {
        const uint32_t a = (uint32_t)__shfl_xor((int)last, (int)o, 64), b = (uint32_t)__shfl_xor((int)begin, (int)o, 64);
        last = a > last ? a : last;
        begin = b < begin ? b : begin;
    }
    last = (uint32_t)__builtin_amdgcn_readfirstlane((int)last);
    begin = (uint32_t)__builtin_amdgcn_readfirstlane((int)begin);
    SmallDraw d0{}, d1{}, n0{}, n1{};
    uint32_t block = 0;  // sweep of the sample block's first slot
    uint32_t k0 = me.k0, k1 = me.k1;
    // sweep it's numbers to n0 and n1
    auto next = [&](uint32_t it) {
        const uint32_t j = it & (B - 1u);
        if (j == 0u) {
            const uint32_t tj = me.t + it + u / W;
            d0 = small_draw(me.acc, k0, k1, w, tj, 0u);
            d1 = small_draw(me.acc, k0, k1, w, tj, 1u);
        }
        const int src = (int)((lane & ~(T - 1u)) + j * W + w);
        auto fetch = [&](const SmallDraw &d) {
            if (B == 1u) return d;
            return SmallDraw{(uint32_t)__shfl((int)d.a1, src, 64), (uint32_t)__shfl((int)d.o1, src, 64),
                             (uint32_t)__shfl((int)d.a2, src, 64), (uint32_t)__shfl((int)d.o2, src, 64),
                             (uint32_t)__shfl((int)d.ranks, src, 64)};
        };
        n0 = fetch(d0);
        n1 = fetch(d1);
    };
    if (last > 0u) next(0u);
    for (uint32_t it = 0; it < last; ++it) {
        // the keys anew in every sweep: their 18 round keys are not kept
        asm volatile("" : "+v"(k0), "+v"(k1));
        const uint32_t t = me.t + it;
        const SmallDraw e0 = n0, e1 = n1;
        // the next sweep's while this one is decided
        next(it + 1u);
        const bool running = it < total;
        {
            const Nbr4 nb = cb_neighbours_small(c1, lane_prev<W>(c1), lane_next<W>(c1), L, 0u);
            const uint32_t f = small_decide(e0, c0, nb, me.acc, k0, k1, w, t, 0u);
            c0 ^= running ? f : 0u;
        }
        {
            const Nbr4 nb = cb_neighbours_small(c0, lane_prev<W>(c0), lane_next<W>(c0), L, 1u);
            const uint32_t f = small_decide(e1, c1, nb, me.acc, k0, k1, w, t, 1u);
            c1 ^= running ? f : 0u;
        }
        if (it < begin) continue;
        if (it == begin) block = it;
        const uint32_t slot = it - block;
        if (u < W) {
            snap[slot * stride + w] = c0;
            snap[slot * stride + W + w] = c1;
        }
        if (slot + 1u < T && it + 1u < last) continue;
        // ---- a block of samples: lane u measures sweep block + u
        small_sync();
        const uint32_t mine = block + u;
        bool pending = me.alive && u <= slot && mine >= me.therm && mine < total;
        const uint32_t bin = pending ? (me.n_measured + (mine - me.therm)) / me.spb : 0u;
        int32_t S[NLMAX + 1u][3], M;
        {
            const uint32_t ts = me.t + mine;
            constexpr uint32_t N1 = SmallLevel<L / 2u>::N;
            uint32_t coin[(N1 + 3u) & ~3u];
            auto draw = [&](uint32_t call, uint32_t level, uint32_t *out) {
                const u32x4 x = philox(call, ts, 0u, (kTagTie << 28) | (level << 16), k0, k1);
                out[0] = x.v0;
                out[1] = x.v1;
                out[2] = x.v2;
                out[3] = x.v3;
            };
#pragma unroll
            for (uint32_t k = 0; 4u * k < N1; ++k) draw(k, 0u, coin + 4u * k);
            const SmallLevel<L / 2u> a = small_level0<L>(snap + u * stride, coin, S[0], M);
            small_levels<L / 2u, 1u, NLMAX>(a, nl, S, draw);
        }
        while (__ballot(pending) != 0ull) {
            // the earliest bin of the team's pending samples
            const uint64_t pend = __ballot(pending) & team;
            const uint32_t from = pend ? (uint32_t)__builtin_ctzll(pend) : lane;
            const uint32_t nb = (uint32_t)__shfl((int)bin, (int)from, 64);
            const bool change = pend != 0ull && nb != rec_bin;
            if (__ballot(change && rec_bin != 0xFFFFFFFFu) != 0ull) flush(change && rec_bin != 0xFFFFFFFFu);
            if (change) rec_bin = nb;
            const bool take = pending && bin == nb;
            small_accumulate<NLMAX>(rec, S, M, take, nl, T, u == 0u);
            pending = pending && !take;
        }
        block = it + 1u;
        small_sync();
    }
    flush(me.alive && rec_bin != 0xFFFFFFFFu);
}

}  // namespace mcrg
