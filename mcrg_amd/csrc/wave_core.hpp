// Lattices of L = 64 and 128 in the registers of one wave.
//
// Lane l holds row l (L = 64) or rows 2l and 2l + 1 (L = 128) of both colours,
// as checkerboard words: 1 or 4 words a colour.  Rows above and below come from
// DPP wave rotations, so a sweep touches neither LDS nor a barrier, and the four
// words of L = 128 keep four random-number chains in flight.
// A sample is measured in two steps.  At once, in registers: the operators of
// the levels down to side 32 (64 x 64 rows of two words, 32 x 32 rows at the
// even lanes) and the blocking to side 16, whose 16 rows go to LDS with the
// counts.  Once 64 sweeps have passed, lane u finishes sample u by itself as in
// small_core.hpp: the levels from side 16 down and the record's terms.
//
// Bound by VALU issue on a filled device (L = 128: 4096 lattices 4420 measured
// updates/ns, 5930 unmeasured) and by a wave's latency below one wave a SIMD
// (5.7 us a measured sweep, 2.2 at L = 64).  Workgroups of four waves with the
// lattice in LDS, the first of which worked off every sample's small levels
// while the others waited, reached 2100 and 3580, and 7.6 us (6.9 at L = 64).
#pragma once

#include "small_core.hpp"

namespace mcrg {

// Levels down to side 32 (0 .. kFront - 1) are counted in the first step, two
// words each; then 8 words of the side-16 level; an odd stride.
template <uint32_t L>
struct WaveGeom {
    static constexpr uint32_t WPL = L == 128u ? 4u : 1u;     // words per lane and colour
    static constexpr uint32_t front = L == 128u ? 3u : 2u;   // first level of side 16
    static constexpr uint32_t NLMAX = L == 128u ? 6u : 5u;
    static constexpr uint32_t stride = 2u * front + 9u;
};

__host__ __device__ inline uint32_t wave_lds_words(uint32_t L, uint32_t nl)
{
    return 64u * (L == 128u ? WaveGeom<128u>::stride : WaveGeom<64u>::stride) + 2u * record_size(nl);
}

// Value of the next (previous) lane of the wave, wrapping.
__device__ __forceinline__ uint32_t wave_next(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x134, 0xF, 0xF, false);  // wave_rol:1
}
__device__ __forceinline__ uint32_t wave_prev(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x13C, 0xF, 0xF, false);  // wave_ror:1
}
// The neighbours' side word of a row word o: `side` is the row's word that
// holds the wrap-around site, p the parity (y + c) & 1.
__device__ __forceinline__ uint32_t row_right(uint32_t o, uint32_t side, bool p) { return p ? (o >> 1) | (side << 31) : o; }
__device__ __forceinline__ uint32_t row_left(uint32_t o, uint32_t side, bool p) { return p ? o : (o << 1) | (side >> 31); }

// One colour's half-sweep: own ^= flips; t the sweep, c the colour.
template <uint32_t L>
__device__ __forceinline__ void wave_half(uint32_t (&own)[WaveGeom<L>::WPL], const uint32_t (&oth)[WaveGeom<L>::WPL],
                                          uint32_t c, const Accept &acc, uint32_t k0, uint32_t k1, uint32_t t)
{
    const uint32_t l = threadIdx.x & 63u;
    if constexpr (L == 64u) {
        const bool p = ((l + c) & 1u) != 0u;
        const uint32_t o = oth[0];
        own[0] ^= metropolis_word(own[0], wave_prev(o), wave_next(o), row_left(o, o, p), row_right(o, o, p), 0xFFFFFFFFu,
                                  acc, k0, k1, l, t, c);
    } else {
        const uint32_t up[2] = {wave_prev(oth[2]), wave_prev(oth[3])}, dn[2] = {wave_next(oth[0]), wave_next(oth[1])};
        uint32_t f[4];
        metropolis_words<4u, 1u, false>(f, acc, k0, k1, t, c, 4u * l, [&](uint32_t k) {
            const uint32_t a = k >> 1, q = k & 1u, o = oth[k], side = oth[k ^ 1u];
            const bool p = ((a + c) & 1u) != 0u;
            return MetropolisSites{own[k], a ? oth[q] : up[q], a ? dn[q] : oth[2u + q],
                                   row_left(o, side, p), row_right(o, side, p)};
        });
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) own[k] ^= f[k];
    }
}

// Operator counts of one word of colour c: s its sites, nu, nd, nl, nr its
// neighbours' words, nx the own-colour word of the row below and nxs that
// row's word with the wrap-around site.
__device__ __forceinline__ void word_ops(uint32_t s, uint32_t nu, uint32_t nd, uint32_t nl, uint32_t nr, uint32_t nx,
                                         uint32_t nxs, bool p, uint32_t c, uint32_t &dnn, uint32_t &dnnn, uint32_t &dp,
                                         uint32_t &down)
{
    const uint32_t dr = row_right(nx, nxs, p), dl = row_left(nx, nxs, p);
    if (c == 0u) dnn += (uint32_t)(popc(s ^ nu) + popc(s ^ nd) + popc(s ^ nl) + popc(s ^ nr));
    dnnn += (uint32_t)(popc(s ^ dr) + popc(s ^ dl));
    dp += (uint32_t)popc(xor3(s, nr, nd) ^ dr);
    down += (uint32_t)popc(s);
}

// Counts summed over the wave, packed in pairs (each at most 32768), into LDS
// by lane 0.
__device__ __forceinline__ void put_counts(uint32_t *out, uint32_t a, uint32_t b, uint32_t c, uint32_t d)
{
    const uint32_t x = group_sum(a | (b << 16), 64u), y = group_sum(c | (d << 16), 64u);
    if ((threadIdx.x & 63u) == 0u) {
        out[0] = x;
        out[1] = y;
    }
}

__device__ __forceinline__ uint32_t majority(uint32_t b1, uint32_t b2, uint32_t b3, uint32_t b4, uint32_t coin)
{
    const uint32_t maj3 = (b1 & b2 & (b3 | b4)) | (b3 & b4 & (b1 | b2));
    const uint32_t tie = ~(xor3(b1, b2, b3) ^ b4) & ~(b1 & b2 & b3 & b4) & (b1 | b2 | b3 | b4);
    return maj3 | (tie & coin);
}

// A level of 32 rows of 32 sites, row l / 2 in each even lane: its counts to
// cnt[0..1] and, when the sample is blocked further, the 16 rows of level
// lv + 1 to w16 (8 words).  coin(call, level) draws four tie-coin words.
template <typename Coin>
__device__ __forceinline__ void rows32(uint32_t row, uint32_t lv, uint32_t nl, Coin coin, uint32_t *cnt, uint32_t *w16)
{
    const uint32_t l = __lane_id();
    const uint32_t d = wave_next(wave_next(row)), r = (row >> 1) | (row << 31), g = (d >> 1) | (d << 31);
    const uint32_t on = (l & 1u) ? 0u : 0xFFFFFFFFu;
    put_counts(cnt, (uint32_t)(popc((row ^ r) & on) + popc((row ^ d) & on)),
               (uint32_t)(popc((row ^ g) & on) + popc((r ^ d) & on)), (uint32_t)popc((xor3(row, r, d) ^ g) & on), 0u);
    if (nl == lv) return;
    // row l / 4 at every fourth lane, coin word l / 8
    const u32x4 x = coin(l >> 5, lv);
    const uint32_t b16 = block16(row, d, (pick4(x, (l >> 3) & 3u) >> (16u * ((l >> 2) & 1u))) & 0xFFFFu);
    if ((l & 3u) == 0u) reinterpret_cast<uint16_t *>(w16)[l >> 2] = (uint16_t)b16;
}

// A level of 64 rows of 64 sites, row l (lo, hi) in each lane: its counts to
// cnt[0..1], then as rows32 with the counts of level lv + 1 to cnt[2..3].
template <typename Coin>
__device__ __forceinline__ void rows64(uint32_t lo, uint32_t hi, uint32_t lv, uint32_t nl, Coin coin, uint32_t *cnt,
                                       uint32_t *w16)
{
    const uint32_t l = __lane_id();
    const uint32_t dlo = wave_next(lo), dhi = wave_next(hi);
    const uint32_t rlo = (lo >> 1) | (hi << 31), rhi = (hi >> 1) | (lo << 31);
    const uint32_t glo = (dlo >> 1) | (dhi << 31), ghi = (dhi >> 1) | (dlo << 31);
    put_counts(cnt, (uint32_t)(popc(lo ^ rlo) + popc(hi ^ rhi) + popc(lo ^ dlo) + popc(hi ^ dhi)),
               (uint32_t)(popc(lo ^ glo) + popc(hi ^ ghi) + popc(rlo ^ dlo) + popc(rhi ^ dhi)),
               (uint32_t)(popc(xor3(lo, rlo, dlo) ^ glo) + popc(xor3(hi, rhi, dhi) ^ ghi)), 0u);
    if (nl == lv) return;
    // rows l / 2 at the even lanes: coin word l / 2
    const u32x4 x = coin(l >> 3, lv);
    const uint32_t cw = pick4(x, (l >> 1) & 3u);
    rows32(block16(lo, dlo, cw & 0xFFFFu) | (block16(hi, dhi, cw >> 16) << 16), lv + 1u, nl, coin, cnt + 2, w16);
}

// The sample's first step: counts of the front levels and the side-16 level
// into out (WaveGeom<L>::stride words).
template <uint32_t L>
__device__ __forceinline__ void wave_sample(const uint32_t (&c0)[WaveGeom<L>::WPL], const uint32_t (&c1)[WaveGeom<L>::WPL],
                                            uint32_t nl, uint32_t t, uint32_t k0, uint32_t k1, uint32_t *out)
{
    const uint32_t l = threadIdx.x & 63u;
    uint32_t dnn = 0, dnnn = 0, dp = 0, down = 0;
    auto coin = [&](uint32_t call, uint32_t level) {
        return philox(call, t, 0u, (kTagTie << 28) | (level << 16), k0, k1);
    };
    if constexpr (L == 64u) {
        const bool p = (l & 1u) != 0u;  // parity of colour 0
        const uint32_t a = c0[0], b = c1[0], an = wave_next(a), bn = wave_next(b);
        word_ops(a, wave_prev(b), bn, row_left(b, b, p), row_right(b, b, p), an, an, p, 0u, dnn, dnnn, dp, down);
        word_ops(b, 0u, an, 0u, row_right(a, a, !p), bn, bn, !p, 1u, dnn, dnnn, dp, down);
        put_counts(out, dnn, dnnn, dp, down);
        if (nl == 0u) return;
        // coin word by = l / 2 of level 0
        const u32x4 x = coin(l >> 3, 0u);
        rows32(majority(a, b, an, bn, pick4(x, (l >> 1) & 3u)), 1u, nl, coin, out + 2, out + 2u * WaveGeom<L>::front);
    } else {
        uint32_t n0[2], n1[2];
#pragma unroll
        for (uint32_t q = 0; q < 2u; ++q) {
            n0[q] = wave_next(c0[q]);
            n1[q] = wave_next(c1[q]);
        }
#pragma unroll
        for (uint32_t a = 0; a < 2u; ++a) {
#pragma unroll
            for (uint32_t q = 0; q < 2u; ++q) {
                const uint32_t k = 2u * a + q, ks = 2u * a + (q ^ 1u);
                const bool p = a != 0u;  // parity of colour 0 in row 2l + a
                const uint32_t nx0 = a ? n0[q] : c0[2u + q], nx0s = a ? n0[q ^ 1u] : c0[2u + (q ^ 1u)];
                const uint32_t nx1 = a ? n1[q] : c1[2u + q], nx1s = a ? n1[q ^ 1u] : c1[2u + (q ^ 1u)];
                word_ops(c0[k], a ? c1[q] : wave_prev(c1[2u + q]), nx1, row_left(c1[k], c1[ks], p),
                         row_right(c1[k], c1[ks], p), nx0, nx0s, p, 0u, dnn, dnnn, dp, down);
                word_ops(c1[k], 0u, nx0, 0u, row_right(c0[k], c0[ks], !p), nx1, nx1s, !p, 1u, dnn, dnnn, dp, down);
            }
        }
        put_counts(out, dnn, dnnn, dp, down);
        if (nl == 0u) return;
        // level 1: 64 rows of 64 sites, row l; coin words 2l, 2l + 1
        const u32x4 x = coin(l >> 1, 0u);
        rows64(majority(c0[0], c1[0], c0[2], c1[2], (l & 1u) ? x.v2 : x.v0),
               majority(c0[1], c1[1], c0[3], c1[3], (l & 1u) ? x.v3 : x.v1), 1u, nl, coin, out + 2,
               out + 2u * WaveGeom<L>::front);
    }
}

// Adds the samples with `take` to the partial record; the terms are at most
// 2^30 (L <= 128) and are summed over the wave in two parts of 20 and 12 bits.
template <uint32_t NLMAX>
__device__ __forceinline__ void wave_accumulate(int64_t *rec, const int32_t (&S)[NLMAX + 1u][3], int32_t M, bool take,
                                                uint32_t nl)
{
    const uint32_t self = 3u * (nl + 1u), cross = 12u * (nl + 1u), nn0 = cross + 9u * nl, tail = nn0 + nl;
    const bool first = (threadIdx.x & 63u) == 0u;
    auto add = [&](uint32_t k, int32_t v) {
        v = take ? v : 0;
        const uint32_t lo = group_sum((uint32_t)v & 0xFFFFFu, 64u);
        const int32_t hi = (int32_t)group_sum((uint32_t)(v >> 20), 64u);
        if (first)
            __hip_atomic_fetch_add(reinterpret_cast<unsigned long long *>(rec + k),
                                   (unsigned long long)(((int64_t)hi << 20) + (int64_t)lo), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
    };
#pragma unroll
    for (uint32_t l = 0; l <= NLMAX; ++l) {
        if (l > nl) break;
#pragma unroll
        for (uint32_t b = 0; b < 3u; ++b) {
            add(3u * l + b, S[l][b]);
#pragma unroll
            for (uint32_t a = 0; a <= b; ++a) add(self + 9u * l + 3u * b + a, S[l][a] * S[l][b]);
            if (l > 0u) {
#pragma unroll
                for (uint32_t a = 0; a < 3u; ++a) add(cross + 9u * (l - 1u) + 3u * b + a, S[l][a] * S[l - (l > 0u)][b]);
            }
        }
        if (l > 0u) add(nn0 + l - 1u, S[l][0] * S[0][0]);
    }
    add(tail, M);
    add(tail + 1u, M < 0 ? -M : M);
    add(tail + 2u, M * M);
    add(tail + 3u, 1);
}

// A block of samples, one a lane with `pending`: the rest of the sample of
// sweep ts, whose entry is `in`, to the record of its bin.  rec holds the record
// of rec_bin (0xFFFFFFFF: none), flush adds it to the results and clears it.
template <uint32_t L, typename Flush>
__device__ __forceinline__ void wave_finish(const uint32_t *in, uint32_t nl, uint32_t k0, uint32_t k1, uint32_t ts,
                                            uint32_t bin, bool pending, int64_t *rec, uint32_t &rec_bin, Flush flush)
{
    using Geom = WaveGeom<L>;
    int32_t S[Geom::NLMAX + 1u][3], M = 0;
#pragma unroll
    for (uint32_t l = 0; l < Geom::front; ++l) {
        const uint32_t x = in[2u * l], y = in[2u * l + 1u];
        const int32_t sites = (int32_t)((L >> l) * (L >> l));
        S[l][0] = 2 * sites - 2 * (int32_t)(x & 0xFFFFu);
        S[l][1] = 2 * sites - 2 * (int32_t)(x >> 16);
        S[l][2] = sites - 2 * (int32_t)(y & 0xFFFFu);
        if (l == 0u) M = sites - 2 * (int32_t)(y >> 16);
    }
    if (nl >= Geom::front) {
        SmallLevel<16u> x;
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) x.w[k] = in[2u * Geom::front + k];
        small_levels<16u, Geom::front, Geom::NLMAX>(x, nl, S, [&](uint32_t call, uint32_t level, uint32_t *out) {
            const u32x4 c = philox(call, ts, 0u, (kTagTie << 28) | (level << 16), k0, k1);
            out[0] = c.v0;
            out[1] = c.v1;
            out[2] = c.v2;
            out[3] = c.v3;
        });
    }
    for (uint64_t pend; (pend = __ballot(pending)) != 0ull;) {
        // the earliest bin of the pending samples
        const uint32_t nb = (uint32_t)__builtin_amdgcn_readlane((int)bin, (int)__builtin_ctzll(pend));
        if (nb != rec_bin) {
            if (rec_bin != 0xFFFFFFFFu) flush();
            rec_bin = nb;
        }
        const bool take = pending && bin == nb;
        wave_accumulate<Geom::NLMAX>(rec, S, M, take, nl);
        pending = pending && !take;
    }
}

// Advances the wave's lattice by up to n sweeps; `me` is the same in every lane.
template <uint32_t L>
__device__ __forceinline__ void run_wave(const SmallLattice &me, uint32_t n, uint32_t nl, uint32_t *lds,
                                         uint32_t (&c0)[WaveGeom<L>::WPL], uint32_t (&c1)[WaveGeom<L>::WPL])
{
    using Geom = WaveGeom<L>;
    const uint32_t u = threadIdx.x & 63u, rs = record_size(nl);
    int64_t *rec = reinterpret_cast<int64_t *>(lds + 64u * Geom::stride);
    for (uint32_t k = u; k < rs; k += 64u) rec[k] = 0;
    uint32_t rec_bin = 0xFFFFFFFFu;  // the bin that rec holds
    auto flush = [&]() {
        small_sync();
        for (uint32_t k = u; k < rs; k += 64u) me.records[(size_t)rec_bin * rs + k] += rec[record_canon(nl, k)];
        small_sync();
        for (uint32_t k = u; k < rs; k += 64u) rec[k] = 0;
        small_sync();
    };
    Accept acc;
    acc.thr0 = uni<true>(me.acc.thr0);
    acc.thr1 = uni<true>(me.acc.thr1);
    acc.always0 = uni<true>(me.acc.always0);
    acc.always1 = uni<true>(me.acc.always1);
    const uint32_t total = uni<true>(me.therm + me.meas), last = total < n ? total : n, therm = uni<true>(me.therm);
    const uint32_t t0 = uni<true>(me.t);
    uint32_t kv0 = me.k0, kv1 = me.k1;
    uint32_t block = therm;  // sweep of the sample block's first slot
    for (uint32_t it = 0; it < last; ++it) {
        // the keys anew in every sweep: their 18 round keys are not kept
        asm volatile("" : "+v"(kv0), "+v"(kv1));
        const uint32_t k0 = uni<true>(kv0), k1 = uni<true>(kv1), t = t0 + it;
        wave_half<L>(c0, c1, 0u, acc, k0, k1, t);
        wave_half<L>(c1, c0, 1u, acc, k0, k1, t);
        if (it < therm) continue;
        const uint32_t slot = it - block;
        wave_sample<L>(c0, c1, nl, t, k0, k1, lds + slot * Geom::stride);
        if (slot + 1u < 64u && it + 1u < last) continue;
        // ---- a block of samples: lane u finishes sweep block + u
        small_sync();
        const uint32_t q0 = me.n_measured + (block - therm);
        wave_finish<L>(lds + u * Geom::stride, nl, k0, k1, t0 + block + u, (q0 + u) / me.spb, u <= slot, rec, rec_bin,
                       flush);
        block = it + 1u;
        small_sync();
    }
    if (rec_bin != 0xFFFFFFFFu) flush();
}

}  // namespace mcrg
