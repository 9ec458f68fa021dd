// Lattices of L = 256 and 512 in a workgroup's LDS: Metropolis sweeps and the
// measurement of every level, for one part of a slot (one lattice).
//
// Checkerboard words of both colours in LDS, four words a thread at a time
// (metropolis_words).  Per measured sweep, a barrier after each:
//   colour 0; colour 1 with the tie coins of the large blockings;
//   level 0 and the blockings down to side 64: each wave its band of rows, with
//   the counts into the sample's entry of a ring;
// and the operators of the levels between, spread over the workgroup.
// Once each wave has a sample, it counts that one's levels of side 64 and 32 in
// registers (rows64) and leaves the 16 x 16 level in the ring; once 64 samples
// are there, wave 0's lane u finishes sample u: the levels from side 16 down and
// the record's terms.  So no wave works on a small level while others wait.
//
// Bound by VALU issue (Philox) where lattices fill the device, and by the
// phases' latency where one has a compute unit to itself (a measured sweep's
// level 0 2.0 us of 16.5, level 1 2.0, the others 1.2).  us a sweep, unmeasured
// and measured, against one word at a time and every level in each sample's
// turn: one L = 512, 1024 threads 14.1 -> 11.5 and 20.9 -> 16.5; 512 of them, 512
// threads 32.5 -> 27.5 and 41.3 -> 30.7; 1024 of L = 256, 256 threads 18.0 ->
// 14.6 and 22.8 -> 19.0.  With level 0 a word at a time and wave 0 alone on sides
// 64 and 32 the first measured sweep took 17.3 and the second 35.
#pragma once

#include "wave_core.hpp"

namespace mcrg {

struct BigLayout {
    uint32_t W, ls;       // words per colour; levels 0 .. ls - 1 are spread (side > 64)
    uint32_t lvl_words;   // words of levels 1 .. min(ls, nl), and of their tie coins
    uint32_t coin_calls;  // Philox calls for those
    uint32_t row64;       // level ls of a sample a wave
    uint32_t stride;      // ring entry: 4 counts a spread level, 2 packed words for
                          // sides 64 and 32 each, 8 words of side 16; odd
    uint32_t spins, lvl, coin, ring, rec, total;
};

__host__ __device__ inline BigLayout big_layout(uint32_t L, uint32_t nl, uint32_t threads)
{
    BigLayout b;
    b.W = cb_words(L);
    b.ls = L == 512u ? 3u : 2u;
    b.lvl_words = 0;
    b.coin_calls = 0;
    for (uint32_t l = 1; l <= b.ls && l <= nl; ++l) {
        b.lvl_words += level_words(L, l);
        b.coin_calls += (level_words(L, l) + 3u) / 4u;
    }
    b.stride = 4u * b.ls + 13u;
    b.spins = 0;
    b.lvl = 2u * b.W;
    b.coin = b.lvl + b.lvl_words;
    b.row64 = b.coin + b.lvl_words;
    b.ring = b.row64 + (nl >= b.ls ? threads / 64u * 128u : 0u);
    b.rec = (b.ring + 64u * b.stride + 1u) & ~1u;
    b.total = b.rec + 2u * record_size(nl);
    return b;
}

// Adds one level's terms of the lanes with `take` to the record: S its
// operators, P those of the level before, nn0 the NN of level 0.  Terms are at
// most 2^38 (L <= 512) and are summed over the wave in two parts.
__device__ __forceinline__ void big_add_level(int64_t *rec, uint32_t nl, uint32_t l, const int32_t (&S)[3],
                                              const int32_t (&P)[3], int32_t nn0, bool take)
{
    const bool first = __lane_id() == 0u;
    auto add = [&](uint32_t k, int64_t v) {
        v = take ? v : 0;
        const uint32_t lo = group_sum((uint32_t)v & 0xFFFFFu, 64u);
        const int32_t hi = (int32_t)group_sum((uint32_t)(v >> 20), 64u);
        if (first)
            __hip_atomic_fetch_add(reinterpret_cast<unsigned long long *>(rec + k),
                                   (unsigned long long)(((int64_t)hi << 20) + (int64_t)lo), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
        __builtin_amdgcn_sched_barrier(0);
    };
    const uint32_t self = 3u * (nl + 1u) + 9u * l, cross = 12u * (nl + 1u) + 9u * (l - 1u);
#pragma unroll
    for (uint32_t b = 0; b < 3u; ++b) {
        add(3u * l + b, S[b]);
#pragma unroll
        for (uint32_t a = 0; a <= b; ++a) add(self + 3u * b + a, (int64_t)S[a] * S[b]);
    }
    if (l == 0u) return;
#pragma unroll
    for (uint32_t b = 0; b < 3u; ++b)
#pragma unroll
        for (uint32_t a = 0; a < 3u; ++a) add(cross + 3u * b + a, (int64_t)S[a] * P[b]);
    add(12u * (nl + 1u) + 9u * nl + l - 1u, (int64_t)S[0] * nn0);
}

// The levels from l on (x is level l, side Ll), as big_add_level.
template <uint32_t Ll, typename Draw>
__device__ __forceinline__ void big_small_levels(const SmallLevel<Ll> &x, int64_t *rec, uint32_t nl, uint32_t l,
                                                 const int32_t (&P)[3], int32_t nn0, bool take, Draw draw)
{
    if (l > nl) return;
    int32_t S[3];
    x.ops(S);
    big_add_level(rec, nl, l, S, P, nn0, take);
    if constexpr (Ll > 2u) {
        if (l < nl) {
            uint32_t coin[4];
            draw(l, coin);
            big_small_levels<Ll / 2u>(x.block(coin), rec, nl, l + 1u, S, nn0, take, draw);
        }
    }
}

template <int NT, uint32_t L>
__device__ __forceinline__ void run_slot(const Slot sl, const int32_t *__restrict__ slot_lats, PackedLattice *__restrict__ lats,
                         uint32_t *lds)
{
    const int32_t li = (int32_t)uni<true>((uint32_t)slot_lats[sl.first]);
    if (li < 0) return;
    PackedLattice &P = lats[li];
    // what is the same in every lane is kept scalar
    const uint32_t nl = uni<true>((uint32_t)sl.n_levels);
    const BigLayout lay = big_layout(L, nl, (uint32_t)NT);
    constexpr uint32_t W = L * L / 64u, ls = L == 512u ? 3u : 2u;
    const uint32_t rs = record_size(nl);
    uint32_t tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    uint32_t *c0 = lds + lay.spins, *c1 = c0 + W, *lvl = lds + lay.lvl, *coins = lds + lay.coin, *ring = lds + lay.ring;
    uint32_t *row64 = lds + lay.row64;
    constexpr uint32_t NW = (uint32_t)NT / 64u;
    int64_t *rec = reinterpret_cast<int64_t *>(lds + lay.rec);
    Accept acc;
    acc.thr0 = uni<true>(P.acc.thr0);
    acc.thr1 = uni<true>(P.acc.thr1);
    acc.always0 = uni<true>(P.acc.always0);
    acc.always1 = uni<true>(P.acc.always1);
    const uint32_t t0 = uni<true>(P.t), therm = uni<true>(P.therm_left), total = uni<true>(therm + P.meas_left);
    const uint32_t last = min(total, uni<true>(sl.n_sweeps));
    uint32_t kv0 = P.k0, kv1 = P.k1;
    for (uint32_t j = tid; j < 2u * W; j += NT) c0[j] = P.spins[j];
    for (uint32_t k = tid; k < rs; k += NT) rec[k] = 0;
    for (uint32_t j = tid; j < 64u * lay.stride; j += NT) ring[j] = 0u;
    uint32_t rec_bin = 0xFFFFFFFFu;  // wave 0: the bin that rec holds
    auto flush = [&]() {
        const uint32_t lane = __lane_id();
        small_sync();
        for (uint32_t k = lane; k < rs; k += 64u) P.records[(size_t)rec_bin * rs + k] += rec[record_canon(nl, k)];
        small_sync();
        for (uint32_t k = lane; k < rs; k += 64u) rec[k] = 0;
        small_sync();
    };
    __syncthreads();
    for (uint32_t it = 0; it < last; ++it) {
        // the keys and the thread's index anew in every sweep: neither the 18
        // round keys nor the words' addresses are kept through the loop
        uint32_t me = threadIdx.x;
        asm volatile("" : "+v"(kv0), "+v"(kv1), "+v"(me));
        const uint32_t lane = me & 63u;
        const uint32_t k0 = uni<true>(kv0), k1 = uni<true>(kv1), t = t0 + it;
        const bool measuring = it >= therm;
        for (uint32_t c = 0; c < 2u; ++c) {
            uint32_t *own = c ? c1 : c0;
            const uint32_t *oth = c ? c0 : c1;
            auto sites = [&](uint32_t w) {
                const Nbr4 n = cb_neighbours(oth, L, W, w, c);
                return MetropolisSites{own[w], n.nu, n.nd, n.nl, n.nr};
            };
            uint32_t w = me;
            for (; w + 3u * NT < W; w += 4u * NT) {
                uint32_t f[4];
                metropolis_words<4u, (uint32_t)NT, true>(f, acc, k0, k1, t, c, w, [&](uint32_t k) { return sites(w + k * NT); });
#pragma unroll
                for (uint32_t k = 0; k < 4u; ++k) own[w + k * NT] ^= f[k];
            }
            for (; w < W; w += NT) {
                uint32_t f[1];
                metropolis_words<1u, 0u, true>(f, acc, k0, k1, t, c, w, [&](uint32_t) { return sites(w); });
                own[w] ^= f[0];
            }
            if (c == 1u && measuring)
                for (uint32_t cc = me; cc < lay.coin_calls; cc += NT) {
                    // calls of levels 1 .. in turn, all of them whole calls
                    uint32_t l = 0, q = cc, off = 0;
                    while (q >= level_words(L, l + 1u) / 4u) {
                        q -= level_words(L, l + 1u) / 4u;
                        off += level_words(L, l + 1u);
                        ++l;
                    }
                    const u32x4 r = philox(q, t, 0u, (kTagTie << 28) | (l << 16), k0, k1);
                    uint32_t *cw = coins + off + 4u * q;
                    cw[0] = r.v0;
                    cw[1] = r.v1;
                    cw[2] = r.v2;
                    cw[3] = r.v3;
                }
            __syncthreads();
        }
        if (!measuring) continue;
        // ---- level 0, and every blocking down to side 64: a wave's band of rows
        //      is blocked from its own rows alone
        const uint32_t slot = (it - therm) & 63u, block = it - slot;  // block: the ring's first sweep
        uint32_t *entry = ring + slot * lay.stride, *last64 = row64 + (slot % NW) * 128u;
        const uint32_t band = me >> 6;
        auto count = [&](uint32_t l, uint32_t d0, uint32_t d1, uint32_t d2, uint32_t d3) {
            d0 = group_sum(d0, 64u);
            d1 = group_sum(d1, 64u);
            d2 = group_sum(d2, 64u);
            if (l == 0u) d3 = group_sum(d3, 64u);
            if (lane == 0u) {
                atomicAdd(entry + 4u * l, d0);
                atomicAdd(entry + 4u * l + 1u, d1);
                atomicAdd(entry + 4u * l + 2u, d2);
                if (l == 0u) atomicAdd(entry + 3, d3);
            }
        };
        {
            constexpr uint32_t wpr = L / 64u, n = W / 2u / NW;
            uint32_t d0 = 0, d1 = 0, d2 = 0, d3 = 0;
            for (uint32_t k = lane; k < n; k += 64u) {
                const uint32_t i = band * n + k, q = i % wpr, y = i / wpr * 2u;
                cb_rows<2u>(c0, c1, wpr, L - 1u, q, y, nl > 0u, coins + i, lvl + i, d0, d1, d2, d3);
            }
            uint32_t off = 0;
            for (uint32_t l = 1; l < ls && l < nl; ++l) {
                small_sync();
                const uint32_t *src = lvl + off;
                off += level_words(L, l);
                uint32_t *dst = l + 1u < ls ? lvl + off : last64;
                const uint32_t m = level_words(L, l + 1u) / NW;
                for (uint32_t k = lane; k < m; k += 64u)
                    dst[band * m + k] = rm_block_item(src, L >> l, band * m + k, coins[off + band * m + k]);
            }
            count(0u, d0, d1, d2, d3);
        }
        __syncthreads();
        // ---- the operators of the levels down to side 128
        {
            uint32_t off = 0;
            for (uint32_t l = 1; l < ls && l <= nl; ++l) {
                uint32_t d0 = 0, d1 = 0, d2 = 0;
                for (uint32_t i = me; i < rm_ops_items(L >> l); i += NT) rm_ops_item(lvl + off, L >> l, i, d0, d1, d2);
                count(l, d0, d1, d2, 0u);
                off += level_words(L, l);
            }
        }
        // ---- a sample a wave: sides 64 and 32, the side-16 level into the ring.
        //      The next sample's levels are written two barriers from here.
        const bool full = slot + 1u == 64u || it + 1u == last;
        if (nl >= ls && (full || slot % NW + 1u == NW)) {
            const uint32_t mine = slot - slot % NW + (me >> 6);
            if (mine <= slot) {
                const uint32_t ts = t0 + block + mine, *row = row64 + (me >> 6) * 128u + 2u * lane;
                auto coin = [&](uint32_t call, uint32_t level) {
                    return philox(call, ts, 0u, (kTagTie << 28) | (level << 16), k0, k1);
                };
                uint32_t *e = ring + mine * lay.stride + 4u * ls;
                rows64(row[0], row[1], ls, nl, coin, e, e + 4u);
            }
        }
        if (full) __syncthreads();
        if (me >= 64u || !full) continue;
        // ---- 64 samples: lane u finishes sweep block + u
        small_sync();
        bool pending = lane <= slot;
        const uint32_t bin = (P.n_measured + (block - therm) + lane) / (uint32_t)P.sweeps_per_bin, ts = t0 + block + lane;
        const uint32_t *in = ring + lane * lay.stride;
        for (uint64_t pend; (pend = __ballot(pending)) != 0ull;) {
            const uint32_t nb = (uint32_t)__builtin_amdgcn_readlane((int)bin, (int)__builtin_ctzll(pend));
            if (nb != rec_bin) {
                if (rec_bin != 0xFFFFFFFFu) flush();
                rec_bin = nb;
            }
            const bool take = pending && bin == nb, first = lane == 0u;
            pending = pending && !take;
            int32_t S[3] = {0, 0, 0}, Sp[3] = {0, 0, 0}, nn0 = 0;
#pragma unroll 1
            for (uint32_t l = 0; l < ls + 2u && l <= nl; ++l) {
                const int32_t n = (int32_t)((L >> l) * (L >> l));
                const uint32_t *e = in + (l < ls ? 4u * l : 4u * ls + 2u * (l - ls));
                const uint32_t x = e[0], y = e[1], z = e[2];
#pragma unroll
                for (uint32_t a = 0; a < 3u; ++a) Sp[a] = S[a];
                S[0] = 2 * n - 2 * (int32_t)(l < ls ? x : x & 0xFFFFu);
                S[1] = 2 * n - 2 * (int32_t)(l < ls ? y : x >> 16);
                S[2] = n - 2 * (int32_t)(l < ls ? z : y & 0xFFFFu);
                if (l == 0u) nn0 = S[0];
                big_add_level(rec, nl, l, S, Sp, nn0, take);
            }
            if (nl >= ls + 2u) {
                SmallLevel<16u> x;
#pragma unroll
                for (uint32_t k = 0; k < 8u; ++k) x.w[k] = in[4u * ls + 4u + k];
                big_small_levels<16u>(x, rec, nl, ls + 2u, S, nn0, take, [&](uint32_t level, uint32_t *out) {
                    const u32x4 r = philox(0u, ts, 0u, (kTagTie << 28) | (level << 16), k0, k1);
                    out[0] = r.v0;
                    out[1] = r.v1;
                    out[2] = r.v2;
                    out[3] = r.v3;
                });
            }
            const int32_t M = take ? (int32_t)(L * L) - 2 * (int32_t)in[3] : 0;
            const int64_t mm = (int64_t)M * M;
            const int32_t m = (int32_t)group_sum((uint32_t)M, 64u), ma = (int32_t)group_sum((uint32_t)(M < 0 ? -M : M), 64u);
            const uint32_t lo = group_sum((uint32_t)mm & 0xFFFFFu, 64u), hi = group_sum((uint32_t)(mm >> 20), 64u);
            const uint32_t count = group_sum(take ? 1u : 0u, 64u);
            if (first) {
                int64_t *tail = rec + 12u * (nl + 1u) + 10u * nl;
                tail[0] += m;
                tail[1] += ma;
                tail[2] += ((int64_t)hi << 20) + (int64_t)lo;
                tail[3] += count;
            }
        }
        small_sync();
        for (uint32_t j = lane; j < 64u * lay.stride; j += 64u) ring[j] = 0u;
    }
    tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    if (tid < 64u && rec_bin != 0xFFFFFFFFu) flush();
    __syncthreads();
    for (uint32_t j = tid; j < 2u * W; j += NT) P.spins[j] = c0[j];
    if (tid == 0u) {
        const uint32_t measured = last > therm ? last - therm : 0u;
        P.t = t0 + last;
        P.n_measured += measured;
        P.therm_left = therm - (last - measured);
        P.meas_left = total - therm - measured;
    }
    __syncthreads();
}

}  // namespace mcrg
