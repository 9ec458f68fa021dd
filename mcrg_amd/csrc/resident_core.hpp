// Pieces shared by the kernels that hold whole lattices (resident_body.hpp,
// wave_core.hpp, small_core.hpp, sw_kernels.hip): wave sums, the record's entry
// list, and the register pyramid of blocked levels.
#pragma once

#include "levels.hpp"
#include "resident.hpp"

namespace mcrg {

// LDS words that several waves read and write between barriers.
__device__ __forceinline__ uint32_t lds_ld(const uint32_t *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_st(uint32_t *p, uint32_t v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Sum over the aligned group of `width` lanes (1..64, a power of two) that
// contains this lane; for width 64 the total is valid in lanes 0..31.
__device__ __forceinline__ uint32_t group_sum(uint32_t v, uint32_t width)
{
    if (width >= 2u) v += (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, false);  // quad_perm 1,0,3,2
    if (width >= 4u) v += (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, false);  // quad_perm 2,3,0,1
    if (width >= 8u) v += (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xF, 0xF, false); // row_half_mirror
    if (width >= 16u) v += (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x140, 0xF, 0xF, false); // row_mirror
    if (width >= 32u) v += (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, 0x401F);             // xor 16
    if (width >= 64u) v += (uint32_t)__builtin_amdgcn_readlane((int)v, 32);
    return v;
}

// Record entry k of one sample is sv[x] * sv[y] over the lattice's operator
// values sv = (S[0][0..2], ..., S[nl][0..2], M, |M|, 1) (layout of record_size():
// S, SELF, CROSS, NN0, then M, |M|, M^2 and the count).
__device__ __forceinline__ void record_pair(uint32_t nl, uint32_t k, uint32_t &x, uint32_t &y)
{
    const uint32_t n_s = 3u * (nl + 1u), n_self = 9u * (nl + 1u), n_cross = 9u * nl, n_nn0 = nl;
    const uint32_t iM = n_s, iAbs = n_s + 1u, iOne = n_s + 2u;
    if (k < n_s) {
        x = k;
        y = iOne;
    } else if (k < n_s + n_self) {
        const uint32_t kk = k - n_s, l = kk / 9u, r = kk % 9u;
        x = 3u * l + r % 3u;
        y = 3u * l + r / 3u;
    } else if (k < n_s + n_self + n_cross) {
        const uint32_t kk = k - n_s - n_self, l = kk / 9u + 1u, r = kk % 9u;
        x = 3u * l + r % 3u;
        y = 3u * (l - 1u) + r / 3u;
    } else if (k < n_s + n_self + n_cross + n_nn0) {
        x = 3u * (k - n_s - n_self - n_cross + 1u);  // NN of level l
        y = 0u;                                       // NN of level 0
    } else {
        const uint32_t m = k - n_s - n_self - n_cross - n_nn0;
        x = m == 0u ? iM : m == 1u ? iAbs : m == 2u ? iM : iOne;
        y = m == 2u ? iM : iOne;
    }
}

// A value that is the same in every lane (UNIFORM), as a scalar.
template <bool UNIFORM>
__device__ __forceinline__ uint32_t uni(uint32_t v)
{
    return UNIFORM ? (uint32_t)__builtin_amdgcn_readfirstlane((int)v) : v;
}

// Row y+1 (mod Ll) for lane y.  A team of a whole wave rotates the wave by one
// lane with DPP (no LDS round trip) and patches the wrap-around row; smaller
// teams shuffle within their segment.
__device__ __forceinline__ uint32_t row_next(uint32_t v, uint32_t y, uint32_t Ll, uint32_t width)
{
    if (width == 64u) {
        const uint32_t n = (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x134, 0xF, 0xF, false);  // wave_rol:1
        const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)v, 0);
        return y == Ll - 1u ? first : n;
    }
    return (uint32_t)__shfl((int)v, (int)((y + 1u) & (Ll - 1u)), (int)width);
}

// Levels pl..nl of one lattice in registers: lane y (< 64, within the team's
// first wave) holds row y of the current level (rows of 64 bits in two words).
// The row below comes from row_next; lane 2by forms blocked row by from its own
// row and the row below, and one shuffle moves it to lane by.  Per level the
// NN and NNN counts travel packed in one register (each < 2^14 for rows of at
// most 64 sites) and are summed with DPP.  `width` is the shuffle segment (the
// team, or 64 when the team spans waves).
__device__ __forceinline__ void pyramid(const uint32_t *lg, const uint32_t *cg, uint32_t *cntg, uint32_t L,
                                        uint32_t pl, uint32_t nl, uint32_t lvl_off, uint32_t coin_off,
                                        uint32_t y, uint32_t width)
{
    uint32_t Ll = L >> pl;
    uint32_t lo = 0, hi = 0;
    if (y < Ll) {
        if (Ll == 64u) {
            lo = lg[lvl_off + 2u * y];
            hi = lg[lvl_off + 2u * y + 1u];
        } else {
            lo = rm_row_small(lg + lvl_off, Ll, y);
        }
    }
    uint32_t coff = coin_off;
    for (uint32_t l = pl; l <= nl; ++l) {
        const bool wide = Ll == 64u;
        const uint32_t Lb = Ll >> 1;
        // coin word of the blocks this lane forms (lane 2by forms blocked row by)
        uint32_t coin = 0;
        if (l < nl && y < Ll && (y & 1u) == 0u) {
            const uint32_t bm = (y >> 1) * Lb;
            coin = cg[coff + (bm >> 5)] >> (bm & 31u);
        }
        // ---- operators of level l
        const uint32_t dlo = row_next(lo, y, Ll, width);
        const uint32_t dhi = wide ? row_next(hi, y, Ll, width) : 0u;
        uint32_t nn_nnn = 0, dp = 0;
        if (y < Ll) {
            if (wide) {
                const uint32_t rlo = (lo >> 1) | (hi << 31), rhi = (hi >> 1) | (lo << 31);
                const uint32_t glo = (dlo >> 1) | (dhi << 31), ghi = (dhi >> 1) | (dlo << 31);
                const uint32_t dnn = (uint32_t)(popc(lo ^ rlo) + popc(hi ^ rhi) + popc(lo ^ dlo) + popc(hi ^ dhi));
                const uint32_t dnnn =
                    (uint32_t)(popc(lo ^ glo) + popc(hi ^ ghi) + popc(rlo ^ dlo) + popc(rhi ^ dhi));
                nn_nnn = dnn | (dnnn << 16);
                dp = (uint32_t)(popc(xor3(lo, rlo, dlo) ^ glo) + popc(xor3(hi, rhi, dhi) ^ ghi));
            } else {
                const uint32_t r = Ll == 32u ? ((lo >> 1) | (lo << 31)) : rot_right_small(lo, Ll);
                const uint32_t g = Ll == 32u ? ((dlo >> 1) | (dlo << 31)) : rot_right_small(dlo, Ll);
                nn_nnn = (uint32_t)(popc(lo ^ r) + popc(lo ^ dlo)) | ((uint32_t)(popc(lo ^ g) + popc(r ^ dlo)) << 16);
                dp = (uint32_t)popc(xor3(lo, r, dlo) ^ g);
            }
        }
        // rows y >= Ll contribute nothing: sum over the level's Ll lanes
        nn_nnn = group_sum(nn_nnn, Ll);
        dp = group_sum(dp, Ll);
        if (y == 0u) {
            uint32_t *c = cntg + l * 4u;
            c[0] = nn_nnn & 0xFFFFu;
            c[1] = nn_nnn >> 16;
            c[2] = dp;
            c[3] = 0u;
        }
        if (l == nl) break;
        // ---- blocking into level l + 1
        uint32_t blk = 0;
        if (y < Ll && (y & 1u) == 0u) {
            if (wide)
                blk = block16(lo, dlo, coin & 0xFFFFu) | (block16(hi, dhi, coin >> 16) << 16);
            else
                blk = block16(lo, dlo, coin) & ((1u << Lb) - 1u);
        }
        const uint32_t nlo = (uint32_t)__shfl((int)blk, (int)((2u * y) & (width - 1u)), (int)width);
        coff += level_words(L, l + 1u);
        lo = y < Lb ? nlo : 0u;
        hi = 0u;
        Ll = Lb;
    }
}

// pyramid() for a starting row width LP and shuffle segment WIDTH known at
// compile time: its levels are unrolled, so every width test (the group sums,
// the row rotation, the 64-site rows) folds away.  The same operations in the
// same order, so the counts and blocked rows are identical.
template <uint32_t LP, uint32_t WIDTH>
__device__ __forceinline__ void pyramid_t(const uint32_t *lg, const uint32_t *cg, uint32_t *cntg, uint32_t L,
                                          uint32_t pl, uint32_t nl, uint32_t lvl_off, uint32_t coin_off,
                                          uint32_t y)
{
    uint32_t lo = 0, hi = 0;
    if (y < LP) {
        if (LP == 64u) {
            lo = lg[lvl_off + 2u * y];
            hi = lg[lvl_off + 2u * y + 1u];
        } else {
            lo = rm_row_small(lg + lvl_off, LP, y);
        }
    }
    uint32_t coff = coin_off;
#pragma unroll
    for (uint32_t j = 0; (LP >> j) >= 2u; ++j) {
        const uint32_t l = pl + j;
        if (l > nl) break;
        const uint32_t Ll = LP >> j;
        const bool wide = Ll == 64u;
        const uint32_t Lb = Ll >> 1;
        // the coin word of the blocks lane y forms (lane 2by forms blocked row
        // by), loaded by every lane (rows y >= Ll wrap into the level) under a
        // wave-uniform test instead of a lane-divergent one
        uint32_t coin = 0;
        if (l < nl) {
            const uint32_t bm = ((y & (Ll - 1u)) >> 1) * Lb;
            coin = cg[coff + (bm >> 5)] >> (bm & 31u);
        }
        const uint32_t dlo = row_next(lo, y, Ll, WIDTH);
        const uint32_t dhi = wide ? row_next(hi, y, Ll, WIDTH) : 0u;
        uint32_t nn_nnn = 0, dp = 0;
        if (y < Ll) {
            if (wide) {
                const uint32_t rlo = (lo >> 1) | (hi << 31), rhi = (hi >> 1) | (lo << 31);
                const uint32_t glo = (dlo >> 1) | (dhi << 31), ghi = (dhi >> 1) | (dlo << 31);
                const uint32_t dnn = (uint32_t)(popc(lo ^ rlo) + popc(hi ^ rhi) + popc(lo ^ dlo) + popc(hi ^ dhi));
                const uint32_t dnnn =
                    (uint32_t)(popc(lo ^ glo) + popc(hi ^ ghi) + popc(rlo ^ dlo) + popc(rhi ^ dhi));
                nn_nnn = dnn | (dnnn << 16);
                dp = (uint32_t)(popc(xor3(lo, rlo, dlo) ^ glo) + popc(xor3(hi, rhi, dhi) ^ ghi));
            } else {
                const uint32_t r = Ll == 32u ? ((lo >> 1) | (lo << 31)) : rot_right_small(lo, Ll);
                const uint32_t g = Ll == 32u ? ((dlo >> 1) | (dlo << 31)) : rot_right_small(dlo, Ll);
                nn_nnn = (uint32_t)(popc(lo ^ r) + popc(lo ^ dlo)) | ((uint32_t)(popc(lo ^ g) + popc(r ^ dlo)) << 16);
                dp = (uint32_t)popc(xor3(lo, r, dlo) ^ g);
            }
        }
        nn_nnn = group_sum(nn_nnn, Ll);
        dp = group_sum(dp, Ll);
        if (y == 0u) {
            uint32_t *c = cntg + l * 4u;
            c[0] = nn_nnn & 0xFFFFu;
            c[1] = nn_nnn >> 16;
            c[2] = dp;
            c[3] = 0u;
        }
        if (l == nl) break;
        uint32_t blk = 0;
        if (y < Ll && (y & 1u) == 0u) {
            if (wide)
                blk = block16(lo, dlo, coin & 0xFFFFu) | (block16(hi, dhi, coin >> 16) << 16);
            else
                blk = block16(lo, dlo, coin) & ((1u << Lb) - 1u);
        }
        const uint32_t nlo = (uint32_t)__shfl((int)blk, (int)((2u * y) & (WIDTH - 1u)), (int)WIDTH);
        coff += level_words(L, l + 1u);
        lo = y < Lb ? nlo : 0u;
        hi = 0u;
    }
}

}  // namespace mcrg
