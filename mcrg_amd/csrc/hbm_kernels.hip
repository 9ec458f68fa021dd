// HBM-resident schedule: int8 lattices in global memory, one launch per
// half-sweep, then two launches per measurement.  Used for the plain
// single-lattice path and for batches of large lattices (one grid row per
// lattice, blockIdx.y).
//
//   k_int8_init           Philox +-1 start        (Lattice::initialize_random_spins, src/lattice.cpp:33-41)
//   k_int8_half_sweep     checkerboard Metropolis (replaces Wolff, src/ising.cpp:87-149)
//   k_int8_measure0       level-0 NN/NNN/P + M and b=2 majority blocking into a
//                         bit-packed level-1 lattice (src/lattice.cpp:102-120, src/mcrg.cpp:314-348)
//   k_rm_level            one large blocked level: operators and the next
//                         blocking, over a grid (src/mcrg.cpp:80-86, src/lattice.cpp:84-120)
//   k_levels_accumulate   the small levels in one workgroup per lattice, then
//                         the per-sample sums and products into the bin record
//                         (src/mcrg.cpp:72-98)
#include "device_common.hpp"
#include "hbm_kernels.hpp"
#include "levels.hpp"

namespace mcrg {

// ---------------------------------------------------------------- init
__global__ __launch_bounds__(256) void k_int8_init(const HbmLattice *__restrict__ lats)
{
    const HbmLattice &lat = lats[blockIdx.y];
    const uint32_t L = (uint32_t)lat.L;
    const uint32_t n = L * L;
    const uint32_t m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= n) return;
    const u32x4 r = philox(m >> 7, 0u, 0u, kTagInit << 28, lat.k0, lat.k1);
    const uint32_t bit = (pick4(r, (m >> 5) & 3u) >> (m & 31u)) & 1u;
    lat.spins[m] = (int8_t)(1 - 2 * (int)bit);
}

// ---------------------------------------------------------------- sweep
// One thread per word of 32 same-colour sites.  For L >= 64 a word is the
// sites of one colour in a 64-byte run of one row.
__device__ __forceinline__ void load64(const int8_t *p, uint32_t d[16])
{
    const uint4 *v = reinterpret_cast<const uint4 *>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint4 x = v[i];
        d[4 * i + 0] = x.x;
        d[4 * i + 1] = x.y;
        d[4 * i + 2] = x.z;
        d[4 * i + 3] = x.w;
    }
}

__device__ __forceinline__ void store64(int8_t *p, const uint32_t d[16])
{
    uint4 *v = reinterpret_cast<uint4 *>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = make_uint4(d[4 * i], d[4 * i + 1], d[4 * i + 2], d[4 * i + 3]);
}

__device__ __forceinline__ uint32_t sbit(int8_t v) { return ((uint32_t)(uint8_t)v) >> 7; }

__global__ __launch_bounds__(256) void k_int8_half_sweep(const HbmLattice *__restrict__ lats,
                                                         uint32_t t_off, uint32_t colour)
{
    const HbmLattice &lat = lats[blockIdx.y];
    const uint32_t L = (uint32_t)lat.L;
    const uint32_t t = lat.state[0] + t_off;
    const uint32_t w = blockIdx.x * blockDim.x + threadIdx.x;
    const Accept acc = lat.acc;
    int8_t *spins = lat.spins;
    if (L >= 64) {
        // One thread per (strip of R rows, 64-column chunk): it slides a window
        // of row chunks down its strip, so each row is read (R + 2) / R times
        // instead of three.  Only the other colour's bytes of the rows
        // above and below are used, and no thread writes those in this half.
        const uint32_t wpr = L >> 6, sh = (uint32_t)__builtin_ctz(wpr);
        const uint32_t R = half_sweep_rows(L);
        if (w >= (L / R) * wpr) return;
        const uint32_t q = w & (wpr - 1u), y0 = (w >> sh) * R;
        uint32_t U[16], C[16], D[16], E[16];
        load64(spins + (size_t)((y0 - 1u) & (L - 1u)) * L + 64u * q, U);
        load64(spins + (size_t)y0 * L + 64u * q, C);
        load64(spins + (size_t)((y0 + 1u) & (L - 1u)) * L + 64u * q, D);
        for (uint32_t r = 0; r < R; ++r) {
            const uint32_t y = y0 + r;
            // the row after next is fetched while this row is decided
            if (r + 1u < R) load64(spins + (size_t)((y + 2u) & (L - 1u)) * L + 64u * q, E);
            const uint32_t p = (y + colour) & 1u;
            const int8_t *rowbase = spins + (size_t)y * L;
            const uint32_t s = gather_parity(C, p);
            const uint32_t o = gather_parity(C, p ^ 1u);
            const uint32_t nu = gather_parity(U, p);
            const uint32_t nd = gather_parity(D, p);
            // the wrap-around site's byte: the last of the chunk before on
            // p = 0 rows, the first of the chunk after on p = 1 rows
            const uint32_t e = sbit(rowbase[(64u * q + 65u * p - 1u) & (L - 1u)]);
            const uint32_t nr = p == 0u ? o : (o >> 1) | (e << 31);
            const uint32_t nl = p == 0u ? (o << 1) | e : o;
            const uint32_t flip = metropolis_word(s, nu, nd, nl, nr, 0xFFFFFFFFu, acc, lat.k0, lat.k1,
                                                  y * wpr + q, t, colour);
            if (flip) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const uint32_t f0 = (flip >> (2 * i)) & 1u, f1 = (flip >> (2 * i + 1)) & 1u;
                    C[i] ^= ((f0 * 0xFEu) << (8u * p)) | ((f1 * 0xFEu) << (8u * p + 16u));
                }
                store64(spins + (size_t)y * L + 64u * q, C);
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                U[i] = C[i];
                C[i] = D[i];
                D[i] = E[i];
            }
        }
        return;
    }
    // L < 64: a word spans several rows; site-by-site.
    const uint32_t half = L >> 1;
    const uint32_t n_sites = L * half;
    const uint32_t n_words = (n_sites + 31u) >> 5;
    if (w >= n_words) return;
    uint32_t s = 0, nu = 0, nd = 0, nl = 0, nr = 0, valid = 0;
    for (uint32_t j = 0; j < 32u; ++j) {
        const uint32_t m = 32u * w + j;
        if (m >= n_sites) break;
        const uint32_t y = m / half, k = m % half;
        const uint32_t x = 2u * k + ((y + colour) & 1u);
        const uint32_t ym = (y - 1u) & (L - 1u), yp = (y + 1u) & (L - 1u);
        const uint32_t xm = (x - 1u) & (L - 1u), xp = (x + 1u) & (L - 1u);
        valid |= 1u << j;
        s |= sbit(spins[y * L + x]) << j;
        nu |= sbit(spins[ym * L + x]) << j;
        nd |= sbit(spins[yp * L + x]) << j;
        nl |= sbit(spins[y * L + xm]) << j;
        nr |= sbit(spins[y * L + xp]) << j;
    }
    const uint32_t flip = metropolis_word(s, nu, nd, nl, nr, valid, acc, lat.k0, lat.k1, w, t, colour);
    for (uint32_t j = 0; j < 32u; ++j) {
        if (!((flip >> j) & 1u)) continue;
        const uint32_t m = 32u * w + j;
        const uint32_t y = m / half, k = m % half;
        const uint32_t x = 2u * k + ((y + colour) & 1u);
        spins[y * L + x] = (int8_t)(-spins[y * L + x]);
    }
}

// ---------------------------------------------------------------- reductions
__device__ __forceinline__ uint32_t wave_sum(uint32_t v)
{
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Adds the N per-thread counts v[0..N-1] of a 256-thread workgroup into
// dst[0..N-1]: wave sums, then one atomic per counter per workgroup.  Every
// thread of the workgroup calls it.
template <int N>
__device__ __forceinline__ void block_add(unsigned long long *dst, uint32_t (&v)[N])
{
    __shared__ uint32_t part[N][4];
    const uint32_t wave = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = wave_sum(v[k]);
    if ((threadIdx.x & 63u) == 0u) {
#pragma unroll
        for (int k = 0; k < N; ++k) part[k][wave] = v[k];
    }
    __syncthreads();
    if (threadIdx.x < (uint32_t)N) {
        const uint32_t k = threadIdx.x;
        const uint32_t tot = part[k][0] + part[k][1] + part[k][2] + part[k][3];
        if (tot) atomicAdd(dst + k, (unsigned long long)tot);
    }
}

// ---------------------------------------------------------------- level 0
// Disagreement counts: dNN = #{bonds with unequal spins} over the 2L^2 nearest
// bonds, dNNN likewise over the 2L^2 diagonal bonds, dP = #{plaquettes with an
// odd number of -1 spins}, ndown = #{-1 spins}.  Then NN = 2L^2 - 2 dNN,
// NNN = 2L^2 - 2 dNNN, P = L^2 - 2 dP, M = L^2 - 2 ndown.
// Sign bits of 32 int8 spins (bit i = spin x0 + i is -1).
__device__ __forceinline__ uint32_t row_bits32(const int8_t *p)
{
    const uint4 *v = reinterpret_cast<const uint4 *>(p);
    const uint4 a = v[0], b = v[1];
    return sign4(a.x) | (sign4(a.y) << 4) | (sign4(a.z) << 8) | (sign4(a.w) << 12) | (sign4(b.x) << 16) |
           (sign4(b.y) << 20) | (sign4(b.z) << 24) | (sign4(b.w) << 28);
}

// One item per (block row by, 32-column chunk q), L >= 32: the operators of
// the sites of rows 2by and 2by + 1 in the chunk and the 16 blocked spins of
// the chunk, stored as half-word by * (L/32) + q of level 1 (bit offset
// 16 (by * L/32 + q) = by * L/2 + 16 q, as in row-major bits).
__global__ __launch_bounds__(256) void k_int8_measure0(const HbmLattice *__restrict__ lats,
                                                       uint32_t t_off)
{
    const HbmLattice &lat = lats[blockIdx.y];
    const uint32_t L = (uint32_t)lat.L;
    const uint32_t t = lat.state[0] + t_off;
    const int8_t *spins = lat.spins;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t c[4] = {0u, 0u, 0u, 0u};  // dNN, dNNN, dP, ndown
    if (L >= 32) {
        const uint32_t cpr = L >> 5;  // 32-site chunks per row == level-1 half-words per block row
        const uint32_t n_items = (L >> 1) * cpr;
        if (i < n_items) {
            const uint32_t by = i >> __builtin_ctz(cpr), q = i & (cpr - 1u);
            uint32_t a[3], nx[3];
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                const uint32_t y = (2u * by + (uint32_t)r) & (L - 1u);
                const int8_t *rowp = spins + (size_t)y * L;
                a[r] = row_bits32(rowp + 32u * q);
                nx[r] = sbit(rowp[(32u * q + 32u) & (L - 1u)]);
            }
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                // right = s(x+1): the row shifted right by one with the next chunk's first bit.
                const uint32_t s = a[r], d = a[r + 1];
                const uint32_t rt = (s >> 1) | (nx[r] << 31), g = (d >> 1) | (nx[r + 1] << 31);
                c[0] += popc(s ^ rt) + popc(s ^ d);
                c[1] += popc(s ^ g) + popc(rt ^ d);
                c[2] += popc(xor3(s, rt, d) ^ g);
                c[3] += popc(s);
            }
            // coin word i >> 1 of level 0, its half i & 1 (the half-word's bit offset mod 32)
            const uint32_t coin = tie_coin_word(i >> 1, t, 0u, lat.k0, lat.k1) >> (16u * (i & 1u));
            reinterpret_cast<uint16_t *>(lat.lvl)[i] = (uint16_t)block16(a[0], a[1], coin & 0xFFFFu);
        }
    } else {
        // L < 32: one thread per level-1 word, site by site.
        const uint32_t Lb = L >> 1;
        const uint32_t nb = Lb * Lb;
        const uint32_t n_words = (nb + 31u) >> 5;
        if (i < n_words) {
            uint32_t out = 0;
            const uint32_t coin = tie_coin_word(i, t, 0u, lat.k0, lat.k1);
            for (uint32_t j = 0; j < 32u; ++j) {
                const uint32_t bm = 32u * i + j;
                if (bm >= nb) break;
                const uint32_t by = bm / Lb, bx = bm % Lb;
                uint32_t nd = 0;
                for (uint32_t v = 0; v < 2u; ++v) {
                    for (uint32_t u = 0; u < 2u; ++u) {
                        const uint32_t x = 2u * bx + u, y = 2u * by + v;
                        const uint32_t xp = (x + 1u) & (L - 1u), yp = (y + 1u) & (L - 1u);
                        const uint32_t a = sbit(spins[y * L + x]), b = sbit(spins[y * L + xp]);
                        const uint32_t cc = sbit(spins[yp * L + x]), d = sbit(spins[yp * L + xp]);
                        c[0] += (a ^ b) + (a ^ cc);
                        c[1] += (a ^ d) + (b ^ cc);
                        c[2] += a ^ b ^ cc ^ d;
                        c[3] += a;
                        nd += a;
                    }
                }
                const uint32_t bit = nd >= 3u ? 1u : nd <= 1u ? 0u : ((coin >> j) & 1u);
                out |= bit << j;
            }
            lat.lvl[i] = out;
        }
    }
    block_add<4>(lat.sums, c);
}

// Rows a thread of k_int8_operators works off: at most 256 workgroups of 1024
// threads, since each takes a ticket of the same word (12 ns).
static uint32_t operators_rows(uint32_t L)
{
    uint32_t rows = 1u;
    while ((uint64_t)(L / rows) * (L / 16u) > 262144u) rows *= 2u;
    return rows;
}

// The level-0 counts of the lattice as it is, without a blocking: a thread per 16
// columns and `rows` rows (L >= 16) or per site.  Workgroups leave their counts in
// the level scratch, and the one that finishes last adds them up.
// Bound by the launch and the host's wait for it below L = 4096, and by memory
// above (L = 16384 reads 268 MB).
__global__ __launch_bounds__(1024) void k_int8_operators(const HbmLattice *__restrict__ lats, uint32_t rows,
                                                         const uint32_t *__restrict__ error,
                                                         unsigned long long *__restrict__ out)
{
    __shared__ uint32_t sum[4], last;
    if (threadIdx.x < 4u) sum[threadIdx.x] = 0u;
    __syncthreads();
    const HbmLattice &lat = lats[0];
    const uint32_t L = (uint32_t)lat.L, i = blockIdx.x * blockDim.x + threadIdx.x, lane = threadIdx.x & 63u;
    const int8_t *spins = lat.spins;
    uint32_t c[4] = {0u, 0u, 0u, 0u};  // dNN, dNNN, dP, ndown
    if (L >= 16u) {
        const uint32_t cpr = L >> 4, q = i & (cpr - 1u), y0 = (i >> __builtin_ctz(cpr)) * rows;
        const bool on = y0 < L;
        // the chunk to the right sits in a lane of this wave, but for lane 63 of wider rows
        const uint32_t right = cpr >= 64u ? (lane + 1u) & 63u : (lane & ~(cpr - 1u)) | ((q + 1u) & (cpr - 1u));
        const bool outside = cpr > 64u && lane == 63u;
        const int8_t *col = spins + 16u * q, *col_next = spins + ((16u * q + 16u) & (L - 1u));
        auto load = [&](uint32_t y, uint32_t &w, uint32_t &shifted) {
            const size_t at = (size_t)(y & (L - 1u)) * L;
            uint4 v = make_uint4(0u, 0u, 0u, 0u);
            if (on) v = *reinterpret_cast<const uint4 *>(col + at);
            uint32_t b = 0;
            if (on && outside) b = sbit(col_next[at]);
            w = sign4(v.x) | (sign4(v.y) << 4) | (sign4(v.z) << 8) | (sign4(v.w) << 12);
            const uint32_t n = (uint32_t)__shfl((int)w, (int)right, 64);
            shifted = (w >> 1) | ((outside ? b : n & 1u) << 15);
        };
        uint32_t s, rt;
        load(y0, s, rt);
        for (uint32_t r = 0; r < rows; ++r) {
            uint32_t d, g;
            load(y0 + r + 1u, d, g);
            c[0] += popc(s ^ rt) + popc(s ^ d);
            c[1] += popc(s ^ g) + popc(rt ^ d);
            c[2] += popc(xor3(s, rt, d) ^ g);
            c[3] += popc(s);
            s = d;
            rt = g;
        }
    } else if (i < L * L) {
        const uint32_t x = i & (L - 1u), y = i / L, xp = (x + 1u) & (L - 1u), yp = (y + 1u) & (L - 1u);
        const uint32_t a = sbit(spins[y * L + x]), b = sbit(spins[y * L + xp]);
        const uint32_t e = sbit(spins[yp * L + x]), d = sbit(spins[yp * L + xp]);
        c[0] = (a ^ b) + (a ^ e);
        c[1] = (a ^ d) + (b ^ e);
        c[2] = a ^ b ^ e ^ d;
        c[3] = a;
    }
    auto add = [&]() {
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) {
            c[k] = wave_sum(c[k]);
            if (lane == 0u) atomicAdd(sum + k, c[k]);
        }
        __syncthreads();
    };
    add();
    if (gridDim.x > 1u) {
        if (threadIdx.x < 4u)
            __hip_atomic_store(lat.lvl + 4u * blockIdx.x + threadIdx.x, sum[threadIdx.x], __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (threadIdx.x == 0u) {
            __threadfence();
            last = atomicAdd(lat.sums + kSumTicket, 1ull) + 1ull == (unsigned long long)gridDim.x ? 1u : 0u;
            __threadfence();
        }
        __syncthreads();
        if (last == 0u) return;
        // at most 256 workgroups: one a thread (sums at most 2^29)
        if (threadIdx.x < 4u) sum[threadIdx.x] = 0u;
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k)
            c[k] = threadIdx.x < gridDim.x ? __hip_atomic_load(lat.lvl + 4u * threadIdx.x + k, __ATOMIC_RELAXED,
                                                               __HIP_MEMORY_SCOPE_AGENT)
                                           : 0u;
        __syncthreads();
        add();
        if (threadIdx.x == 0u) lat.sums[kSumTicket] = 0ull;
    }
    if (threadIdx.x < kOperatorWords)
        __hip_atomic_store(out + threadIdx.x,
                           (unsigned long long)(threadIdx.x < 4u ? sum[threadIdx.x] : error ? *error : 0u),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---------------------------------------------------------------- levels >= 1
// A grid-measured level l (side Ll >= kGridLevelMinL): one thread per word of
// the level for its operators, and one per word of level l + 1 for the
// blocking when l < nl (ties take the coin words of level l).
__global__ __launch_bounds__(256) void k_rm_level(const HbmLattice *__restrict__ lats, uint32_t level,
                                                  uint32_t t_off)
{
    const HbmLattice &lat = lats[blockIdx.y];
    const uint32_t L = (uint32_t)lat.L;
    const uint32_t t = lat.state[0] + t_off;
    const uint32_t Ll = L >> level;
    const uint32_t *src = lat.lvl + level_offset(L, level);
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t c[3] = {0u, 0u, 0u};
    if (i < rm_ops_items(Ll)) rm_ops_item(src, Ll, i, c[0], c[1], c[2]);
    if (level < (uint32_t)lat.n_levels && i < rm_block_items(Ll))
        lat.lvl[level_offset(L, level + 1u) + i] = rm_block_item(src, Ll, i, tie_coin_word(i, t, level, lat.k0, lat.k1));
    block_add<3>(lat.sums + 4u + 3u * (level - 1u), c);
}

constexpr uint32_t kLevelsThreads = 512;

// Disagreement counts of one RM level, summed over the workgroup into cnt[0..2].
__device__ void rm_ops(const uint32_t *buf, uint32_t Ll, uint32_t *cnt)
{
    uint32_t dnn = 0, dnnn = 0, dp = 0;
    const uint32_t n = rm_ops_items(Ll);
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) rm_ops_item(buf, Ll, i, dnn, dnnn, dp);
    dnn = wave_sum(dnn);
    dnnn = wave_sum(dnnn);
    dp = wave_sum(dp);
    if ((threadIdx.x & 63u) == 0u) {
        atomicAdd(cnt + 0, dnn);
        atomicAdd(cnt + 1, dnnn);
        atomicAdd(cnt + 2, dp);
    }
}

// b = 2 majority blocking of an RM level (size Ll) into dst (size Ll/2).
__device__ void rm_block(const uint32_t *src, uint32_t Ll, uint32_t *dst, uint32_t t,
                         uint32_t level, uint32_t k0, uint32_t k1)
{
    const uint32_t n_out = rm_block_items(Ll);
    for (uint32_t i = threadIdx.x; i < n_out; i += blockDim.x)
        dst[i] = rm_block_item(src, Ll, i, tie_coin_word(i, t, level, k0, k1));
}

// One workgroup per lattice: the levels below kGridLevelMinL (the first read
// from global memory, the deeper ones in LDS), then the operator values of
// every level (grid-measured levels and level 0 from the counters, which it
// clears) and the sample's terms added to its bin record, one entry per thread.
__global__ __launch_bounds__(kLevelsThreads) void k_levels_accumulate(const HbmLattice *__restrict__ lats,
                                                                      uint32_t t_off, uint32_t q_off)
{
    const HbmLattice &lat = lats[blockIdx.x];
    const uint32_t L = (uint32_t)lat.L;
    const uint32_t nl = (uint32_t)lat.n_levels;
    const uint32_t t = lat.state[0] + t_off;
    const uint32_t l0 = n_grid_levels(L, nl) + 1u;  // first level of this workgroup
    __shared__ uint32_t cnt[kMaxLevels + 1][3];
    __shared__ uint32_t bufA[level_words(kWgLevelMaxL / 2u)];
    __shared__ uint32_t bufB[level_words(kWgLevelMaxL / 4u)];
    __shared__ int64_t S[kMaxLevels + 1][3];
    __shared__ int64_t Msh;
    for (uint32_t i = threadIdx.x; i < (kMaxLevels + 1) * 3; i += blockDim.x) (&cnt[0][0])[i] = 0u;
    __syncthreads();
    if (l0 <= nl) {
        const uint32_t *cur = lat.lvl + level_offset(L, l0);
        uint32_t Ll = L >> l0;
        for (uint32_t l = l0; l <= nl; ++l) {
            rm_ops(cur, Ll, cnt[l]);
            if (l < nl) {
                uint32_t *dst = ((l - l0) & 1u) ? bufB : bufA;
                __syncthreads();
                rm_block(cur, Ll, dst, t, l, lat.k0, lat.k1);
                __syncthreads();
                cur = dst;
                Ll >>= 1;
            }
        }
    }
    __syncthreads();
    // operator values; every counter is read and cleared by one thread
    const uint32_t n_s = 3u * (nl + 1u);
    for (uint32_t i = threadIdx.x; i <= n_s; i += blockDim.x) {
        if (i == n_s) {
            Msh = (int64_t)L * L - 2 * (int64_t)lat.sums[3];
            lat.sums[3] = 0ull;
            continue;
        }
        const uint32_t l = i / 3u, a = i % 3u;
        const int64_t nlv = (int64_t)(L >> l) * (L >> l);
        int64_t d;
        if (l == 0u || l < l0) {
            unsigned long long *sp = l == 0u ? lat.sums + a : lat.sums + 4u + 3u * (l - 1u) + a;
            d = (int64_t)*sp;
            *sp = 0ull;
        } else {
            d = cnt[l][a];
        }
        S[l][a] = (a == 2u ? nlv : 2 * nlv) - 2 * d;
    }
    __syncthreads();
    const uint32_t q = lat.state[1] + q_off;
    const uint32_t bin = q / (uint32_t)lat.sweeps_per_bin;
    const uint32_t rs = record_size(nl);
    int64_t *rec = lat.records + (size_t)bin * rs;
    for (uint32_t j = threadIdx.x; j < rs; j += blockDim.x) rec[j] += record_term(j, nl, S, Msh);
}

// Advances the chain's sweep counter and sample counter after a chunk.
__global__ void k_advance(const HbmLattice *__restrict__ lats, uint32_t n_lats, uint32_t sweeps,
                          uint32_t samples)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_lats) return;
    lats[i].state[0] += sweeps;
    lats[i].state[1] += samples;
}

// ---------------------------------------------------------------- launchers
static inline uint32_t cdiv(uint32_t a, uint32_t b) { return (a + b - 1u) / b; }

hipError_t launch_int8_init(const HbmLattice *d, int n_lats, int L, hipStream_t s)
{
    const uint32_t n = (uint32_t)L * (uint32_t)L;
    hipLaunchKernelGGL(k_int8_init, dim3(cdiv(n, 256u), (uint32_t)n_lats), dim3(256), 0, s, d);
    return hipGetLastError();
}

hipError_t launch_int8_half_sweep(const HbmLattice *d, int n_lats, int L, uint32_t t_off,
                                  uint32_t colour, hipStream_t s)
{
    const uint32_t n_sites = (uint32_t)L * (uint32_t)L / 2u;
    const uint32_t n_words = cdiv(n_sites, 32u);
    // L >= 64: one thread per strip of half_sweep_rows(L) rows and 64 columns
    const uint32_t n_items = L >= 64 ? n_words / half_sweep_rows((uint32_t)L) : n_words;
    hipLaunchKernelGGL(k_int8_half_sweep, dim3(cdiv(n_items, 256u), (uint32_t)n_lats), dim3(256), 0,
                       s, d, t_off, colour);
    return hipGetLastError();
}

hipError_t launch_int8_operators(const HbmLattice *d, int L, const uint32_t *error, unsigned long long *out,
                                 hipStream_t s)
{
    const uint32_t rows = operators_rows((uint32_t)L), n = (uint32_t)L;
    const uint32_t n_items = n >= 16u ? n / rows * (n / 16u) : n * n;
    const uint32_t threads = n_items >= 1024u ? 1024u : 256u;  // 256: one workgroup
    hipLaunchKernelGGL(k_int8_operators, dim3(cdiv(n_items, threads)), dim3(threads), 0, s, d, rows, error, out);
    return hipGetLastError();
}

hipError_t launch_int8_measure0(const HbmLattice *d, int n_lats, int L, uint32_t t_off,
                                hipStream_t s)
{
    const uint32_t Lb = (uint32_t)L / 2u;
    const uint32_t n_items = L >= 32 ? Lb * ((uint32_t)L / 32u) : cdiv(Lb * Lb, 32u);
    hipLaunchKernelGGL(k_int8_measure0, dim3(cdiv(n_items, 256u), (uint32_t)n_lats), dim3(256), 0,
                       s, d, t_off);
    return hipGetLastError();
}

hipError_t launch_levels_accumulate(const HbmLattice *d, int n_lats, int L, int n_levels, uint32_t t_off,
                                    uint32_t q_off, hipStream_t s)
{
    const uint32_t g = n_grid_levels((uint32_t)L, (uint32_t)n_levels);
    for (uint32_t l = 1; l <= g; ++l) {
        const uint32_t Ll = (uint32_t)L >> l;
        hipLaunchKernelGGL(k_rm_level, dim3(cdiv(Ll * (Ll / 32u), 256u), (uint32_t)n_lats), dim3(256), 0, s, d,
                           l, t_off);
    }
    hipLaunchKernelGGL(k_levels_accumulate, dim3((uint32_t)n_lats), dim3(kLevelsThreads), 0, s, d, t_off,
                       q_off);
    return hipGetLastError();
}

hipError_t launch_advance(const HbmLattice *d, int n_lats, uint32_t sweeps, uint32_t samples,
                          hipStream_t s)
{
    hipLaunchKernelGGL(k_advance, dim3(cdiv((uint32_t)n_lats, 64u)), dim3(64), 0, s, d,
                       (uint32_t)n_lats, sweeps, samples);
    return hipGetLastError();
}

}  // namespace mcrg
