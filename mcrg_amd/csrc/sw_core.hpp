// Swendsen-Wang building blocks on bit-packed rows in LDS, shared by the
// one-workgroup and the tiled kernels.
//
// Stream: right and down bonds of the site pair (2p, 2p+1) from
// Philox(p, t, 0, 4<<28) (v0, v1 of site 2p, v2, v3 of site 2p+1); the coin of
// the cluster whose smallest site is m is bit m & 127 of Philox(m>>7, t, 0, 5<<28).
//
// A block of words (the whole lattice, or a 64 x 64 tile) holds row-major bits:
// 32 sites a word, rows of less than 32 sites sharing words.  A run is a
// maximal set of sites of one row joined by right bonds inside one word; its
// first site stands for it.  Run starts, ends and fills come from bit
// arithmetic, so 31/32 of the right bonds and half of the sites never enter the
// union-find, and a thread works off a part of PW sites of a word (PW = 32 where
// many lattices or tiles fill the device, fewer where one lattice has it alone).
//
// Labels (LDS, one per site, used at run starts only) are padded site ids,
// m + m/32, so that the words of a wave's lanes lie in different banks.  The
// forest points to smaller ids only; ids are in site order, so each tree's root
// is the smallest site of its cluster whatever the order of the unions.
#pragma once

#include "hbm_kernels.hpp"
#include "resident_core.hpp"

namespace mcrg {

// Unions a wave gathers before it works them off.
constexpr uint32_t kSwList = 256;

__device__ __forceinline__ uint32_t sw_id(uint32_t m) { return m + (m >> 5); }
__device__ __forceinline__ uint32_t sw_site(uint32_t id) { return id - id / 33u; }

__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Set bits of v below this lane.
__device__ __forceinline__ uint32_t mbcnt(uint64_t v)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(v >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)v, 0u));
}

// OR over the aligned group of 32 / PW lanes that shares a word.
template <uint32_t PW>
__device__ __forceinline__ uint32_t word_or(uint32_t v)
{
#pragma unroll
    for (uint32_t o = 1; o < 32u / PW; o <<= 1) v |= (uint32_t)__shfl_xor((int)v, (int)o, 64);
    return v;
}

// The uniforms' comparisons of the PW sites from site pair p on: right (r) and
// down (d) bonds drawn, bit k for the part's site k.  32-bit words of the whole
// group after word_or.
template <uint32_t PW>
__device__ __forceinline__ void sw_draw(uint32_t p, uint32_t t, uint32_t thr, uint32_t k0, uint32_t k1, uint32_t &r,
                                        uint32_t &d)
{
    r = d = 0;
#pragma unroll 2
    for (uint32_t k = PW / 2u; k-- > 0u;) {
        const u32x4 x = philox(p + k, t, 0u, kTagSwBond << 28, k0, k1);
        r = (r << 2) | (x.v2 < thr ? 2u : 0u) | (x.v0 < thr ? 1u : 0u);
        d = (d << 2) | (x.v3 < thr ? 2u : 0u) | (x.v1 < thr ? 1u : 0u);
    }
}

// First site of the run of bonds r that bit b belongs to.
__device__ __forceinline__ uint32_t run_start(uint32_t r, uint32_t b)
{
    const uint32_t z = ~r & ((1u << b) - 1u);
    return z ? 32u - (uint32_t)__builtin_clz(z) : 0u;
}

// Bits that have a bit of g before them in their run (bond b of r joins bits b
// and b + 1).
__device__ __forceinline__ uint32_t run_later(uint32_t g, uint32_t r)
{
    uint32_t p = r;
#pragma unroll
    for (uint32_t o = 1; o < 32u; o <<= 1) {
        g |= (g & p) << o;
        p &= p >> o;
    }
    return (g & r) << 1;
}

// Joins the trees of a and b, walking up both at once and halving the paths
// (every second label on the way moves to its parent's parent, so that the
// chains that simultaneous links leave behind shrink under the walks); of two
// roots the larger is linked below the smaller.  A label is smaller than its own
// id (but a root's) and always names a site of the same cluster, so a stale read
// lengthens a path but never leaves the cluster.  A halving store that comes late
// may raise a label that another thread's fetch_min has just lowered; that thread
// then unites the old label's tree itself, since fetch_min gave it that label.
__device__ __forceinline__ void lds_unite(uint32_t *lab, uint32_t a, uint32_t b)
{
    for (;;) {
        const uint32_t pa = lds_ld(lab + a), pb = lds_ld(lab + b);
        if (pa == pb) return;
        if (pa != a || pb != b) {
            const uint32_t ga = lds_ld(lab + pa), gb = lds_ld(lab + pb);
            if (ga != pa) lds_st(lab + a, ga);
            if (gb != pb) lds_st(lab + b, gb);
            a = ga;
            b = gb;
            continue;
        }
        const uint32_t lo = a < b ? a : b, hi = a < b ? b : a;
        const uint32_t old = __hip_atomic_fetch_min(lab + hi, lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (old == hi) return;
        // hi stopped being a root: go on from what it was linked to
        a = lo;
        b = old;
    }
}

// Bits of a word's part.
template <uint32_t PW>
__device__ __forceinline__ uint32_t part_mask(uint32_t lo)
{
    return PW == 32u ? 0xFFFFFFFFu : ((1u << (PW & 31u)) - 1u) << lo;
}

// Labels of the runs that start in `starts` (bits of word i with run bonds r):
// the run above that the run's first bond from above (up) comes from, or the
// run itself.  rup are the run bonds of the row above, aligned with the word;
// site m of the word has m - L above it.  (Rising on up to four rows in
// registers made these first chains shorter but not the walks: L = 64, 16 sites
// a thread, 20.7 -> 22.3 us a sweep.)
__device__ __forceinline__ void sw_hook(uint32_t *lab, uint32_t i, uint32_t L, uint32_t starts, uint32_t r, uint32_t up,
                                        uint32_t rup)
{
    while (starts != 0u) {
        const uint32_t s = (uint32_t)__builtin_ctz(starts);
        starts &= starts - 1u;
        const uint32_t run = (r >> s) ^ ((r >> s) + 1u);  // the run's sites, from bit 0
        const uint32_t f = (up >> s) & run;
        uint32_t label = 33u * i + s;
        if (f != 0u) label = sw_id(32u * i + run_start(rup, s + (uint32_t)__builtin_ctz(f)) - L);
        lds_st(lab + 33u * i + s, label);
    }
}

// The roots of up to four of the runs that start in `starts`, taken off it:
// s[k] their bits (32 where there are fewer) and p[k] the roots' ids.  Paths
// are halved on the way, for the walks beside and behind this one.
__device__ __forceinline__ void sw_roots4(uint32_t *lab, uint32_t i, uint32_t &starts, uint32_t s[4], uint32_t p[4])
{
    uint32_t x[4];
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) {
        s[k] = starts ? (uint32_t)__builtin_ctz(starts) : 32u;
        starts &= starts - 1u;
        x[k] = s[k] < 32u ? 33u * i + s[k] : 0u;  // id 0 is its own root
        p[k] = lds_ld(lab + x[k]);
    }
    for (bool more = true; more;) {
        uint32_t g[4];
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) g[k] = lds_ld(lab + p[k]);
        more = false;
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) {
            if (g[k] == p[k]) continue;
            lds_st(lab + x[k], g[k]);
            x[k] = p[k];
            p[k] = g[k];
            more = true;
        }
    }
}

// Works off the unions of a wave's lanes: bonds from above (`rem`, bits of word
// i, whose runs are r and, in the row above, rup) and links out of the word's
// segments (`link`).  above(b) and next(b) give the padded ids of the run above
// bit b and of the site right of bit b.  They are gathered into full waves,
// four a lane and round, because the lanes' counts differ much.
template <typename Above, typename Next>
__device__ __forceinline__ void sw_unions(uint32_t *lab, uint32_t *list, uint32_t i, uint32_t r, uint32_t rem,
                                          uint32_t link, Above above, Next next)
{
    const uint32_t lane = threadIdx.x & 63u;
    for (;;) {
        uint32_t n = (uint32_t)popc(rem) + (uint32_t)popc(link);
        n = n < 4u ? n : 4u;
        const uint64_t b0 = __ballot((n & 1u) != 0u), b1 = __ballot((n & 2u) != 0u), b2 = __ballot((n & 4u) != 0u);
        const uint32_t total = (uint32_t)(__builtin_popcountll(b0) + 2 * __builtin_popcountll(b1) +
                                          4 * __builtin_popcountll(b2));
        if (total == 0u) return;
        uint32_t at = mbcnt(b0) + 2u * mbcnt(b1) + 4u * mbcnt(b2);
        for (uint32_t k = 0; k < n; ++k, ++at) {
            uint32_t b, other;
            if (rem != 0u) {
                b = (uint32_t)__builtin_ctz(rem);
                rem &= rem - 1u;
                other = above(b);
            } else {
                b = (uint32_t)__builtin_ctz(link);
                link &= link - 1u;
                other = next(b);
            }
            list[at] = (33u * i + run_start(r, b)) | (other << 16);
        }
        wave_sync();
        for (uint32_t j = lane; j < total; j += 64u) {
            const uint32_t ab = list[j];
            lds_unite(lab, ab & 0xFFFFu, ab >> 16);
        }
        wave_sync();
    }
}

// The int8 spins of 32 sites as bits (bit 1 = spin -1), and back.
__device__ __forceinline__ uint32_t sw_load32(const int8_t *p)
{
    const uint4 *v = reinterpret_cast<const uint4 *>(p);
    const uint4 a = v[0], b = v[1];
    return sign4(a.x) | (sign4(a.y) << 4) | (sign4(a.z) << 8) | (sign4(a.w) << 12) | (sign4(b.x) << 16) |
           (sign4(b.y) << 20) | (sign4(b.z) << 24) | (sign4(b.w) << 28);
}

__device__ __forceinline__ void sw_store32(int8_t *p, uint32_t w)
{
    uint32_t d[8];
#pragma unroll
    for (uint32_t k = 0; k < 8u; ++k) {
        const uint32_t x = (w >> (4u * k)) & 15u;
        // bit j of x to byte j: 0xFF for 1, 0x01 for 0
        d[k] = 0x01010101u | (((x | (x << 7) | (x << 14) | (x << 21)) & 0x01010101u) * 0xFEu);
    }
    uint4 *v = reinterpret_cast<uint4 *>(p);
    v[0] = make_uint4(d[0], d[1], d[2], d[3]);
    v[1] = make_uint4(d[4], d[5], d[6], d[7]);
}

}  // namespace mcrg
