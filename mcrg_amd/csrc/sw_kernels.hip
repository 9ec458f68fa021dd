// Swendsen-Wang cluster sweeps: the Wolff construction (src/ising.cpp:96-149)
// for every cluster at once, with union-find on bit-packed bonds (sw_core.hpp).
//
//   k_sw_wg   a whole lattice of L <= kSwWgMaxL in one workgroup's LDS, for all
//             the sweeps of a launch, with the measurement of every level and
//             the records (src/lattice.cpp:102-120, src/mcrg.cpp:72-98, :314-348)
//   k_sw_tile, k_sw_seam, k_sw_apply
//             larger lattices, one sweep in three launches: clusters within
//             64 x 64 tiles, their unions across tiles, the flips
//   k_sw_measure0
//             level-0 operators and the blocking into level 1, from bits
#include <algorithm>

#include "lds_opt_in.hpp"
#include "sw_core.hpp"

namespace mcrg {

// Row-major bits of a lattice of n = L*L sites: site m is bit m & 31 of word
// m >> 5.  A segment is the part of a row inside one word (32 sites, or the row
// when it is shorter); seg_ends marks its last bit.
__device__ __forceinline__ uint32_t seg_ends(uint32_t L)
{
    return L >= 32u ? 0x80000000u : L == 16u ? 0x80008000u : L == 8u ? 0x80808080u : L == 4u ? 0x88888888u : 0xAAAAAAAAu;
}

// Bit b: the right neighbour (same row, periodic) of bit b of word i.
__device__ __forceinline__ uint32_t bits_right(const uint32_t *S, uint32_t L, uint32_t i)
{
    const uint32_t w = S[i];
    if (L >= 32u) {
        const uint32_t wpr = L >> 5;
        return (w >> 1) | (S[(i & ~(wpr - 1u)) | ((i + 1u) & (wpr - 1u))] << 31);
    }
    const uint32_t e = seg_ends(L);
    return ((w >> 1) & ~e) | ((w << (L - 1u)) & e);
}

// Bit b: the site below bit b of word i (periodic).
__device__ __forceinline__ uint32_t bits_down(const uint32_t *S, uint32_t L, uint32_t i)
{
    const uint32_t n = L * L;
    if (L >= 32u) {
        const uint32_t nw = n >> 5, wpr = L >> 5;
        return S[i + wpr < nw ? i + wpr : i + wpr - nw];
    }
    if (n >= 32u) return (S[i] >> L) | (S[(i + 1u) & ((n >> 5) - 1u)] << (32u - L));
    return ((S[i] >> L) | (S[i] << (n - L))) & ((1u << n) - 1u);
}

// Bit b: the site above bit b of word i (periodic).
__device__ __forceinline__ uint32_t bits_up(const uint32_t *S, uint32_t L, uint32_t i)
{
    const uint32_t n = L * L;
    if (L >= 32u) {
        const uint32_t nw = n >> 5, wpr = L >> 5;
        return S[i >= wpr ? i - wpr : i + nw - wpr];
    }
    if (n >= 32u) return (S[i] << L) | (S[(i - 1u) & ((n >> 5) - 1u)] >> (32u - L));
    return ((S[i] << L) | (S[i] >> (n - L))) & ((1u << n) - 1u);
}

struct SwWgLayout {
    uint32_t nw;  // words of the lattice
    uint32_t lvl_words, coin_calls, n_sv;
    uint32_t S, R, D, C, lab, list, lvl, coin, cnt, sv, pairs, rec, total;  // offsets in 32-bit words
};

// `threads` of the workgroup work on the lattice (the measuring wave beside
// them has no list).
__host__ __device__ inline SwWgLayout sw_wg_layout(uint32_t L, uint32_t nl, uint32_t threads)
{
    SwWgLayout s;
    const uint32_t n = L * L;
    s.nw = (n + 31u) / 32u;
    s.lvl_words = 0;
    s.coin_calls = 0;
    for (uint32_t l = 1; l <= nl; ++l) {
        s.lvl_words += level_words(L >> l);
        s.coin_calls += (level_words(L >> l) + 3u) / 4u;
    }
    s.n_sv = 3u * (nl + 1u) + 3u;
    s.lab = 0;
    s.list = s.lab + 33u * s.nw;
    s.S = s.list + threads / 64u * kSwList;
    s.R = s.S + s.nw;
    s.D = s.R + s.nw;
    s.C = s.D + s.nw;
    s.lvl = s.C + ((s.nw + 3u) & ~3u);
    s.coin = s.lvl + s.lvl_words;
    s.cnt = s.coin + 2u * s.lvl_words;
    s.sv = s.cnt + 4u * (nl + 1u);
    s.pairs = s.sv + s.n_sv;
    s.rec = (s.pairs + record_size(nl) + 1u) & ~1u;
    s.total = s.rec + 2u * record_size(nl);
    return s;
}

// Workgroup b advances lats[b] by n sweeps, all measured or none, and its
// counters.  One lattice in LDS: int8 spins are read once and written once per
// launch.  The last wave measures the blocked levels and adds the record terms
// while the others are in the next sweep (tie coins alternate between two
// buffers for it); it may be one more than the lattice's.  Per sweep, a barrier
// after each:
//   bonds    drawn a part at a time and kept as words R (right) and D (down),
//            with the clusters' coin bits and the tie coins
//   hooks    every run labelled with the run above that its first bond from
//            above comes from
//   unions   the remaining bonds from above (a bond whose left neighbour joins
//            the same two runs left out) and the links between segments
//   flips    every run's root and coin, carried along the run by an addition
// Bound by the latency of the walks in the union-find (LDS round trips): a
// measured L = 64 sweep takes 12 us on its own (bonds 1.4, hooks 1.1, unions
// 4.3, flips 3.2, level 0 0.9) against 36 us with a launch per phase, and 1024
// lattices take 23 us against 105.
template <uint32_t PW>
__global__ __launch_bounds__(1024) void k_sw_wg(const HbmLattice *__restrict__ lats, uint32_t n, uint32_t measure,
                                                uint32_t n_work)
{
    extern __shared__ uint32_t lds[];
    const HbmLattice &lat = lats[blockIdx.x];
    const uint32_t L = (uint32_t)lat.L, nl = (uint32_t)lat.n_levels, ns = L * L;
    const SwWgLayout lay = sw_wg_layout(L, nl, n_work);
    uint32_t *lab = lds + lay.lab, *S = lds + lay.S, *R = lds + lay.R, *D = lds + lay.D, *C = lds + lay.C;
    uint32_t *lvl = lds + lay.lvl, *coins = lds + lay.coin, *cnt = lds + lay.cnt, *pairs = lds + lay.pairs;
    int32_t *sv = reinterpret_cast<int32_t *>(lds + lay.sv);
    int64_t *rec = reinterpret_cast<int64_t *>(lds + lay.rec);
    const uint32_t tid = threadIdx.x, NT = blockDim.x, lane = tid & 63u, rs = record_size(nl);
    const uint32_t t0 = lat.state[0], q0 = lat.state[1], spb = (uint32_t)lat.sweeps_per_bin;
    const uint32_t k0 = lat.k0, k1 = lat.k1, thr = lat.bond_thr;
    const uint32_t ends = seg_ends(L), valid = ns >= 32u ? 0xFFFFFFFFu : (1u << ns) - 1u;
    const uint32_t n_parts = lay.nw * (32u / PW);
    const bool work = tid < n_work;
    uint32_t *list = lds + lay.list + (work ? tid >> 6 : 0u) * kSwList;

    for (uint32_t i = tid; i < lay.nw; i += NT) {
        uint32_t w = 0;
        if (ns >= 32u)
            w = sw_load32(lat.spins + 32u * i);
        else
            for (uint32_t j = 0; j < ns; ++j) w |= (((uint32_t)(uint8_t)lat.spins[j]) >> 7) << j;
        S[i] = w;
    }
    for (uint32_t k = tid; k < rs; k += NT) {
        uint32_t x, y;
        record_pair(nl, k, x, y);
        pairs[k] = x | (y << 16);
        rec[k] = 0;
    }
    for (uint32_t i = tid; i < 4u * (nl + 1u); i += NT) cnt[i] = 0u;
    __syncthreads();

    for (uint32_t it = 0; it < n; ++it) {
        const uint32_t t = t0 + it;
        uint32_t *coin = coins + (it & 1u) * lay.lvl_words;
        // ---- bonds
        if (work) {
            // coin bits of the clusters (word m >> 5 of site m) and the sample's
            // tie coins, from the workgroup's last threads on
            const uint32_t n_c = (lay.nw + 3u) / 4u, n_draw = n_c + (measure ? lay.coin_calls : 0u);
            for (uint32_t c = n_work - 1u - tid; c < n_draw; c += n_work) {
                uint32_t l = 0, q = c, off = 0, w = 4u * n_c, tag = kTagSwFlip << 28;
                uint32_t *cw = C;  // padded to whole calls
                if (c >= n_c) {
                    q -= n_c;
                    for (; l + 1u < nl; ++l) {
                        const uint32_t calls = (level_words(L >> (l + 1u)) + 3u) / 4u;
                        if (q < calls) break;
                        q -= calls;
                        off += level_words(L >> (l + 1u));
                    }
                    w = level_words(L >> (l + 1u));
                    tag = (kTagTie << 28) | (l << 16);
                    cw = coin + off;
                }
                const u32x4 r = philox(q, t, 0u, tag, k0, k1);
                cw += 4u * q;
                cw[0] = r.v0;
                if (4u * q + 1u < w) cw[1] = r.v1;
                if (4u * q + 2u < w) cw[2] = r.v2;
                if (4u * q + 3u < w) cw[3] = r.v3;
            }
            for (uint32_t p0 = tid - lane; p0 < n_parts; p0 += n_work) {
                const uint32_t part = p0 + lane, i = part / (32u / PW), lo = part % (32u / PW) * PW;
                uint32_t r, d;
                sw_draw<PW>((32u * i + lo) >> 1, t, thr, k0, k1, r, d);
                r = word_or<PW>(r << lo);
                d = word_or<PW>(d << lo);
                if (lo == 0u && i < lay.nw) {
                    const uint32_t s = S[i];
                    R[i] = r & ~(s ^ bits_right(S, L, i)) & valid;
                    D[i] = d & ~(s ^ bits_down(S, L, i)) & valid;
                }
            }
        }
        __syncthreads();
        // ---- hooks
        if (work)
            for (uint32_t part = tid; part < n_parts; part += n_work) {
                const uint32_t i = part / (32u / PW), lo = part % (32u / PW) * PW;
                const uint32_t row0 = L >= 32u ? (i < (L >> 5) ? 0xFFFFFFFFu : 0u) : i == 0u ? (1u << L) - 1u : 0u;
                const uint32_t r = R[i] & ~ends;
                sw_hook(lab, i, L, ~(r << 1) & part_mask<PW>(lo) & valid, r, bits_up(D, L, i) & ~row0,
                        bits_up(R, L, i) & ~ends);
            }
        __syncthreads();
        // ---- unions
        if (work)
            for (uint32_t p0 = tid - lane; p0 < n_parts; p0 += n_work) {
                const uint32_t part = p0 + lane, i = part / (32u / PW), lo = part % (32u / PW) * PW;
                uint32_t r = 0, rem = 0, link = 0, rup = 0;
                if (part < n_parts) {
                    const uint32_t row0 = L >= 32u ? (i < (L >> 5) ? 0xFFFFFFFFu : 0u) : i == 0u ? (1u << L) - 1u : 0u;
                    const uint32_t up = bits_up(D, L, i), Ri = R[i];
                    r = Ri & ~ends;
                    rup = bits_up(R, L, i) & ~ends;
                    rem = up & ~((up & r & rup) << 1) & (run_later(up & ~row0, r) | row0) & part_mask<PW>(lo);
                    link = Ri & ends & part_mask<PW>(lo);
                }
                sw_unions(
                    lab, list, i, r, rem, link,
                    [&](uint32_t b) {
                        const uint32_t m = 32u * i + run_start(rup, b);
                        return sw_id(m >= L ? m - L : m + ns - L);
                    },
                    [&](uint32_t b) {
                        const uint32_t m = 32u * i + b;
                        return sw_id((m & ~(L - 1u)) | ((m + 1u) & (L - 1u)));
                    });
            }
        __syncthreads();
        // ---- flips
        if (work)
            for (uint32_t p0 = tid - lane; p0 < n_parts; p0 += n_work) {
                const uint32_t part = p0 + lane, i = part / (32u / PW), lo = part % (32u / PW) * PW;
                uint32_t r = 0, f = 0;
                if (part < n_parts) {
                    r = R[i] & ~ends;
                    uint32_t st = ~(r << 1) & part_mask<PW>(lo) & valid, s[4], p[4];
                    while (st != 0u) {
                        sw_roots4(lab, i, st, s, p);
#pragma unroll
                        for (uint32_t k = 0; k < 4u; ++k) {
                            const uint32_t m = sw_site(p[k]);
                            if (s[k] < 32u) f |= ((C[m >> 5] >> (m & 31u)) & 1u) << s[k];
                        }
                    }
                }
                f = word_or<PW>(f);
                // a run's bonds are ones up to its last site, so adding its
                // start's bit turns over exactly the run
                if (lo == 0u && part < n_parts) S[i] ^= (r + f) ^ r;
            }
        __syncthreads();
        if (!measure) continue;
        // ---- level 0 and the blocking into level 1
        {
            uint32_t d0 = 0, d1 = 0, d2 = 0, d3 = 0;
            for (uint32_t i = tid; i < rm_ops_items(L); i += NT) rm_ops_item(S, L, i, d0, d1, d2);
            for (uint32_t i = tid; i < lay.nw; i += NT) d3 += (uint32_t)popc(S[i]);
            if (nl > 0u) {
                const uint32_t w = level_words(L >> 1);
                for (uint32_t i = NT - 1u - tid; i < w; i += NT) lvl[i] = rm_block_item(S, L, i, coin[i]);
            }
            if (tid - lane < rm_ops_items(L)) {  // at least as many as words
                d0 = group_sum(d0, 64u);
                d1 = group_sum(d1, 64u);
                d2 = group_sum(d2, 64u);
                d3 = group_sum(d3, 64u);
                if (lane == 0u) {
                    atomicAdd(cnt + 0, d0);
                    atomicAdd(cnt + 1, d1);
                    atomicAdd(cnt + 2, d2);
                    atomicAdd(cnt + 3, d3);
                }
            }
        }
        __syncthreads();
        // ---- blocked levels, operator values and the record on the last wave
        if (tid + 64u >= NT) {
            if (L == 128u && nl > 0u)
                pyramid_t<64u, 64u>(lvl, coin, cnt, L, 1u, nl, 0u, level_words(L >> 1), lane);
            else if (L == 64u && nl > 0u)
                pyramid_t<32u, 64u>(lvl, coin, cnt, L, 1u, nl, 0u, level_words(L >> 1), lane);
            else if (nl > 0u)
                pyramid(lvl, coin, cnt, L, 1u, nl, 0u, level_words(L >> 1), lane, 64u);
            wave_sync();
            if (lane < lay.n_sv) {  // at most 3 * 7 + 3
                const uint32_t l = lane / 3u, x = lane - 3u * l, sites = (L >> l) * (L >> l);
                const int32_t M = (int32_t)ns - 2 * (int32_t)cnt[3];
                int32_t v = x == 0u ? M : x == 1u ? (M < 0 ? -M : M) : 1;
                if (l <= nl) v = (int32_t)(x == 2u ? sites : 2u * sites) - 2 * (int32_t)cnt[4u * l + x];
                sv[lane] = v;
            }
            wave_sync();
            const uint32_t q = q0 + it;
            const bool new_bin = q % spb == 0u && it > 0u;  // a full bin goes to memory
            for (uint32_t k = lane; k < rs; k += 64u) {
                int64_t v = rec[k];
                if (new_bin) {
                    lat.records[(size_t)((q - 1u) / spb) * rs + k] += v;
                    v = 0;
                }
                const uint32_t xy = pairs[k];
                rec[k] = v + (int64_t)sv[xy & 0xFFFFu] * (int64_t)sv[xy >> 16];
            }
            if (lane < 4u) cnt[lane] = 0u;
        }
    }
    __syncthreads();
    if (measure && n > 0u)
        for (uint32_t k = tid; k < rs; k += NT) lat.records[(size_t)((q0 + n - 1u) / spb) * rs + k] += rec[k];
    for (uint32_t i = tid; i < lay.nw; i += NT) {
        if (ns >= 32u)
            sw_store32(lat.spins + 32u * i, S[i]);
        else
            for (uint32_t j = 0; j < ns; ++j) lat.spins[j] = (int8_t)(1 - 2 * (int)((S[i] >> j) & 1u));
    }
    if (tid == 0u) {
        lat.state[0] = t0 + n;
        lat.state[1] = q0 + (measure ? n : 0u);
    }
}

template <uint32_t PW>
static hipError_t launch_sw_wg_pw(const HbmLattice *d, int n_lats, uint32_t lds_bytes, uint32_t n, bool measure,
                                  uint32_t n_work, uint32_t threads, hipStream_t s)
{
    static LdsOptIn lds;
    const hipError_t le = lds.need(reinterpret_cast<const void *>(&k_sw_wg<PW>), lds_bytes);
    if (le != hipSuccess) return le;
    hipLaunchKernelGGL(k_sw_wg<PW>, dim3((uint32_t)n_lats), dim3(threads), lds_bytes, s, d, n, measure ? 1u : 0u,
                       n_work);
    return hipGetLastError();
}

int sw_wg_part(int n_lats, int L, int n_cus)
{
    // The smallest part whose threads (at most 512 a lattice, at most 1024 a
    // compute unit over all lattices) are there at once: more threads shorten
    // the phases until they wait for each other (L = 64 alone: 8 sites a thread
    // 10.1 us a sweep, 16 14.2, 32 22; 1024 lattices: 16 sites 20.6, 32 26.2).
    const int nw = std::max(1, L * L / 32);
    for (int pw = 4; pw < 32; pw *= 2) {
        const int64_t threads = std::max(64, nw * (32 / pw));
        if (threads <= 512 && threads * n_lats <= (int64_t)1024 * n_cus) return pw;
    }
    return 32;
}

hipError_t launch_sw_wg(const HbmLattice *d, int n_lats, int L, int n_levels, int part, uint32_t n, bool measure,
                        int n_cus, hipStream_t s)
{
    if (L > kSwWgMaxL || part < 4 || part > 32) return hipErrorInvalidValue;
    const uint32_t parts = (uint32_t)(std::max(1, L * L / 32) * (32 / part));
    const uint32_t n_work = std::min(512u, (parts + 63u) / 64u * 64u);
    // The extra wave only where a lattice has a compute unit to itself: of four
    // workgroups of 4 + 1 waves a unit holds three, since each puts two waves on
    // one of the four SIMDs (1024 x L = 64 measured: 32 us a sweep, 24 without).
    const uint32_t threads = n_work + (measure && n_levels > 0 && n_lats <= n_cus ? 64u : 0u);
    const uint32_t lds_bytes =
        sw_wg_lds_bytes(4u * sw_wg_layout((uint32_t)L, (uint32_t)n_levels, n_work).total, n_lats, n_cus);
    switch (part) {
    case 4: return launch_sw_wg_pw<4>(d, n_lats, lds_bytes, n, measure, n_work, threads, s);
    case 8: return launch_sw_wg_pw<8>(d, n_lats, lds_bytes, n, measure, n_work, threads, s);
    case 16: return launch_sw_wg_pw<16>(d, n_lats, lds_bytes, n, measure, n_work, threads, s);
    case 32: return launch_sw_wg_pw<32>(d, n_lats, lds_bytes, n, measure, n_work, threads, s);
    default: return hipErrorInvalidValue;
    }
}

// ------------------------------------------------------------------ tiles
// A tile is 64 x 64 sites, two words a row.  k_sw_tile finds its clusters in
// LDS.  A cluster that reaches none of the tile's edge sites is complete: it is
// flipped there and then.  Each other cluster is a node, named by its largest
// edge position (top 0..63, bottom 64..127, left 128..191, right 192..255); no
// node is named 0, since site (0, 0) is also left position 128, so 0 in the
// site map stands for clusters that are done.  k_sw_seam unites the nodes
// across the tiles' edges, and k_sw_apply flips what is left by its root's coin.
// A node is (parent node, smallest site); roots are linked by their sites, so
// a tree's root holds the smallest site of the cluster.
constexpr uint32_t kTile = 64, kTileWords = 128, kTileSites = 4096, kTileNodes = 256;
constexpr uint32_t kTag = 0x80000000u;  // label of a root that is a node

struct SwTiles {
    uint32_t *bits;    // [L * L / 32] the lattice's row-major bits
    uint32_t *runs;    // [tile][128] run bonds
    uint64_t *nodes;   // [tile][256] parent | site << 32
    uint64_t *seams;   // [tile][2] bonds over the right and the lower edge
    uint8_t *map;      // [tile][4096] node of the run that starts at a site
    uint8_t *edge;     // [tile][256] node of each edge position
};

__host__ __device__ inline size_t sw_tiles_words(uint32_t L)
{
    const size_t n = (size_t)L * L, tiles = n / kTileSites;
    return n / 32u * 2u + tiles * (2u * kTileNodes + 4u + kTileSites / 4u + kTileNodes / 4u);
}

__device__ __forceinline__ SwTiles sw_tiles(const HbmLattice &lat)
{
    const uint32_t L = (uint32_t)lat.L;
    const size_t n = (size_t)L * L, tiles = n / kTileSites;
    SwTiles s;
    s.nodes = reinterpret_cast<uint64_t *>(lat.sw);
    s.seams = s.nodes + tiles * kTileNodes;
    s.bits = reinterpret_cast<uint32_t *>(s.seams + tiles * 2u);
    s.runs = s.bits + n / 32u;
    s.map = reinterpret_cast<uint8_t *>(s.runs + n / 32u);
    s.edge = s.map + tiles * kTileSites;
    return s;
}

// The root of label x in a tile, where roots may carry a tag.
__device__ __forceinline__ uint32_t tile_root(uint32_t *lab, uint32_t x)
{
    uint32_t p = lds_ld(lab + x);
    if (p & kTag) return x;
    for (;;) {
        const uint32_t g = lds_ld(lab + p);
        if (g == p || (g & kTag)) return p;
        lds_st(lab + x, g);
        x = p;
        p = g;
    }
}

// One workgroup per tile (blockIdx.x) and lattice (blockIdx.y), a thread for
// each part of PW sites.  `first`: the spins come from the int8 lattice, else
// from the bits of the sweep before.
// Bound by the latency of the walks in the union-find (14k cycles of 45k for the
// unions, 12k for the runs' roots, alike with four and with six waves a SIMD)
// and by VALU issue (about 70%).  64 lattices of L = 1024: three launches 377 ->
// 347 us a sweep with seven workgroups a compute unit instead of six, one
// comparison a step of a walk instead of three, and every run's label set to
// its root at the end of its walk.
template <uint32_t PW>
__global__ __launch_bounds__(kTileSites / PW) void k_sw_tile(const HbmLattice *__restrict__ lats, uint32_t t_off,
                                                             uint32_t first)
{
    constexpr uint32_t NT = kTileSites / PW;
    // 23040 bytes in all, a multiple of the allocation unit (1280) of which seven
    // workgroups find room in a compute unit: the row below and the column to the
    // right are read before there are labels, and the edge positions' roots take
    // the words of the down bonds, which are in registers by then
    __shared__ uint32_t words[kTileWords + 33u * kTileWords];
    uint32_t *S = words, *lab = words + kTileWords, *col = lab + 2;
    // the lists of unions, later the site map
    constexpr uint32_t kScratch = NT / 64u * kSwList > kTileSites / 4u ? NT / 64u * kSwList : kTileSites / 4u;
    __shared__ __align__(16) uint32_t scratch[kScratch];
    __shared__ uint32_t R[kTileWords], D[kTileWords], C[kTileWords];
    uint16_t *node_root = reinterpret_cast<uint16_t *>(D);
    static_assert(2u * kTileNodes <= sizeof(D), "node_root");
    const HbmLattice &lat = lats[blockIdx.y];
    const uint32_t L = (uint32_t)lat.L, mask = L - 1u, wpr = L >> 5;
    const SwTiles st = sw_tiles(lat);
    const uint32_t tiles_x = L / kTile, tx = blockIdx.x & (tiles_x - 1u), ty = blockIdx.x >> ilog2u(tiles_x);
    const uint32_t x0 = tx * kTile, y0 = ty * kTile, tile = blockIdx.x;
    const uint32_t t = lat.state[0] + t_off, k0 = lat.k0, k1 = lat.k1, thr = lat.bond_thr;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    // ---- spins: the tile's words, the row below it, the column right of it
    if (tid < kTileWords + 2u) {
        const uint32_t y = (y0 + (tid >> 1)) & mask, x = x0 + 32u * (tid & 1u);
        S[tid] = first ? sw_load32(lat.spins + (size_t)y * L + x) : st.bits[y * wpr + (x >> 5)];
    }
    if (NT < kTileWords + 2u && tid < 2u) {
        const uint32_t y = (y0 + kTile) & mask, x = x0 + 32u * tid;
        S[kTileWords + tid] = first ? sw_load32(lat.spins + (size_t)y * L + x) : st.bits[y * wpr + (x >> 5)];
    }
    if (tid < 64u) {
        const uint32_t y = y0 + lane, x = (x0 + kTile) & mask;
        const uint32_t b = first ? ((uint32_t)(uint8_t)lat.spins[(size_t)y * L + x]) >> 7 : st.bits[y * wpr + (x >> 5)];
        const uint64_t c = __ballot((b & 1u) != 0u);
        if (lane < 2u) col[lane] = (uint32_t)(c >> (32u * lane));
        // coin bits of row lane: 128 sites a call, of which the tile has half
        const uint32_t m = y * L + x0;
        const u32x4 r = philox(m >> 7, t, 0u, kTagSwFlip << 28, k0, k1);
        C[2u * lane] = (m & 64u) ? r.v2 : r.v0;
        C[2u * lane + 1u] = (m & 64u) ? r.v3 : r.v1;
    }
    const uint32_t i = tid / (32u / PW), lo = tid % (32u / PW) * PW, row = i >> 1;
    uint32_t dr, dd;
    sw_draw<PW>(((y0 + row) * L + x0 + 32u * (i & 1u) + lo) >> 1, t, thr, k0, k1, dr, dd);
    dr = word_or<PW>(dr << lo);
    dd = word_or<PW>(dd << lo);
    __syncthreads();
    // ---- bonds
    if (lo == 0u) {
        const uint32_t s = S[i];
        const uint32_t next = (i & 1u) ? (col[row >> 5] >> (row & 31u)) : S[i + 1u];
        R[i] = dr & ~(s ^ ((s >> 1) | (next << 31)));
        D[i] = dd & ~(s ^ S[i + 2u]);
    }
    __syncthreads();
    const uint32_t ends = 0x80000000u;
    const uint32_t r = R[i] & ~ends, up = i >= 2u ? D[i - 2u] : 0u, rup = i >= 2u ? R[i - 2u] & ~ends : 0u;
    const uint32_t seam0 = D[kTileWords - 2u], seam1 = D[kTileWords - 1u];
    const uint32_t pm = part_mask<PW>(lo);
    sw_hook(lab, i, kTile, ~(r << 1) & pm, r, up, rup);
    __syncthreads();
    sw_unions(
        lab, scratch + tid / 64u * kSwList, i, r, up & ~((up & r & rup) << 1) & run_later(up, r) & pm,
        (i & 1u) ? 0u : R[i] & ends & pm, [&](uint32_t b) { return 33u * (i - 2u) + run_start(rup, b); },
        [&](uint32_t) { return 33u * (i + 1u); });
    __syncthreads();
    // ---- nodes: the roots of the edge sites, each named by its largest position
    for (uint32_t pos = tid; pos < kTileNodes; pos += NT) {
        const uint32_t k = pos & 63u, side = pos >> 6;
        const uint32_t y = side == 0u ? 0u : side == 1u ? 63u : k, x = side == 2u ? 0u : side == 3u ? 63u : k;
        const uint32_t w = 2u * y + (x >> 5);
        const uint32_t root = tile_root(lab, 33u * w + run_start(R[w] & ~ends, x & 31u));
        __hip_atomic_fetch_max(lab + root, kTag | pos, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        node_root[pos] = (uint16_t)root;
    }
    {
        uint4 *z = reinterpret_cast<uint4 *>(scratch);
        for (uint32_t k = tid; k < kTileSites / 16u; k += NT) z[k] = make_uint4(0u, 0u, 0u, 0u);
    }
    __syncthreads();
    for (uint32_t pos = tid; pos < kTileNodes; pos += NT) {
        const uint32_t root = node_root[pos], id = lds_ld(lab + root) & 0xFFu;
        st.edge[(size_t)tile * kTileNodes + pos] = (uint8_t)id;
        if (id == pos) {
            const uint32_t m = sw_site(root), site = (y0 + (m >> 6)) * L + x0 + (m & 63u);
            st.nodes[(size_t)tile * kTileNodes + pos] =
                (uint64_t)(tile * kTileNodes + pos) | ((uint64_t)site << 32);
        }
    }
    // ---- every run: its node into the map, or its coin
    uint32_t f = 0, starts = ~(r << 1) & pm;
    uint8_t *map = reinterpret_cast<uint8_t *>(scratch);
    while (starts != 0u) {
        uint32_t s[4], p[4], v[4];
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) {
            s[k] = starts ? (uint32_t)__builtin_ctz(starts) : 32u;
            starts &= starts - 1u;
            p[k] = 33u * i + (s[k] & 31u);
            v[k] = lds_ld(lab + p[k]);
        }
        // v is the label of p: less than p unless p is a root (labels point to
        // smaller ids, and a root's is its own or a tag).  A label moves on to
        // its parent's unless that is a root.
        for (;;) {
            if (__ballot(v[0] < p[0] || v[1] < p[1] || v[2] < p[2] || v[3] < p[3]) == 0ull) break;
            uint32_t u[4];
#pragma unroll
            for (uint32_t k = 0; k < 4u; ++k) u[k] = lds_ld(lab + (v[k] < p[k] ? v[k] : p[k]));
#pragma unroll
            for (uint32_t k = 0; k < 4u; ++k) {
                const bool on = v[k] < p[k];
                if (on && u[k] < v[k]) lds_st(lab + p[k], u[k]);
                p[k] = on ? v[k] : p[k];
                v[k] = u[k];
            }
        }
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) {
            if (s[k] >= 32u) continue;
            // for the walks beside and behind this one
            lds_st(lab + 33u * i + s[k], (v[k] & kTag) ? v[k] : p[k]);
            if (v[k] & kTag) {
                map[32u * i + s[k]] = (uint8_t)v[k];
            } else {
                const uint32_t m = sw_site(p[k]);
                f |= ((C[m >> 5] >> (m & 31u)) & 1u) << s[k];
            }
        }
    }
    f = word_or<PW>(f);
    if (lo == 0u) {
        st.bits[(y0 + row) * wpr + (x0 >> 5) + (i & 1u)] = S[i] ^ ((r + f) ^ r);
        st.runs[(size_t)tile * kTileWords + i] = r;
    }
    if (tid < 64u) {
        const uint64_t b = __ballot((R[2u * lane + 1u] & ends) != 0u);
        if (lane == 0u) {
            st.seams[2u * tile] = b;
            st.seams[2u * tile + 1u] = (uint64_t)seam0 | ((uint64_t)seam1 << 32);
        }
    }
    __syncthreads();
    {
        const uint4 *z = reinterpret_cast<const uint4 *>(scratch);
        uint4 *out = reinterpret_cast<uint4 *>(st.map + (size_t)tile * kTileSites);
        for (uint32_t k = tid; k < kTileSites / 16u; k += NT) out[k] = z[k];
    }
}

__device__ __forceinline__ uint64_t node_ld(const uint64_t *nodes, uint32_t x)
{
    return __hip_atomic_load(nodes + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The root of node x and its smallest site, paths halved on the way.
__device__ __forceinline__ uint32_t node_root_of(uint64_t *nodes, uint32_t x, uint32_t &site)
{
    uint64_t e = node_ld(nodes, x);
    for (;;) {
        const uint32_t p = (uint32_t)e;
        if (p == x) {
            site = (uint32_t)(e >> 32);
            return x;
        }
        const uint64_t g = node_ld(nodes, p);
        if ((uint32_t)g != p)
            __hip_atomic_store(reinterpret_cast<uint32_t *>(nodes + x), (uint32_t)g, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        x = p;
        e = g;
    }
}

// One wave per seam: blockIdx.x covers two tiles, waves 0, 1 the first one's
// right and lower edge, 2, 3 the second's.
__global__ __launch_bounds__(256) void k_sw_seam(const HbmLattice *__restrict__ lats)
{
    const HbmLattice &lat = lats[blockIdx.y];
    const uint32_t L = (uint32_t)lat.L;
    const SwTiles st = sw_tiles(lat);
    const uint32_t tiles_x = L / kTile, lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t tile = 2u * blockIdx.x + (wave >> 1);
    const bool down = (wave & 1u) != 0u;
    const uint32_t tx = tile & (tiles_x - 1u), ty = tile >> ilog2u(tiles_x);
    const uint32_t other = down ? (((ty + 1u) & (tiles_x - 1u)) * tiles_x + tx)
                                : (ty * tiles_x + ((tx + 1u) & (tiles_x - 1u)));
    const uint64_t bonds = st.seams[2u * tile + (down ? 1u : 0u)];
    const uint32_t a = st.edge[(size_t)tile * kTileNodes + (down ? 64u : 192u) + lane];
    const uint32_t b = st.edge[(size_t)other * kTileNodes + (down ? 0u : 128u) + lane];
    // a bond that joins the same two nodes as the one before it is left out
    const uint32_t ab = a | (b << 8) | (uint32_t)((bonds >> lane) & 1u) << 16;
    const uint32_t before = (uint32_t)__shfl_up((int)ab, 1, 64);
    if ((ab >> 16) == 0u || (lane > 0u && before == ab)) return;
    uint32_t u = tile * kTileNodes + a, v = other * kTileNodes + b;
    for (;;) {
        uint32_t su, sv;
        u = node_root_of(st.nodes, u, su);
        v = node_root_of(st.nodes, v, sv);
        if (u == v) return;
        const uint32_t lo = su < sv ? u : v;
        uint32_t hi = su < sv ? v : u, expect = hi;
        if (__hip_atomic_compare_exchange_strong(reinterpret_cast<uint32_t *>(st.nodes + hi), &expect, lo,
                                                 __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            return;
        // hi was linked meanwhile
        u = lo;
        v = expect;
    }
}

// One workgroup per tile: the nodes' coins, then the flips of their runs; with
// `last` the spins as int8 as well.
__global__ __launch_bounds__(256) void k_sw_apply(const HbmLattice *__restrict__ lats, uint32_t t_off, uint32_t last)
{
    __shared__ uint8_t flip[kTileNodes];
    const HbmLattice &lat = lats[blockIdx.y];
    const uint32_t L = (uint32_t)lat.L, wpr = L >> 5, tid = threadIdx.x, tile = blockIdx.x;
    const SwTiles st = sw_tiles(lat);
    const uint4 ids = reinterpret_cast<const uint4 *>(st.map + (size_t)tile * kTileSites)[tid];
    const uint32_t r = st.runs[(size_t)tile * kTileWords + (tid >> 1)];
    uint32_t f = 0;
    if (tid > 0u && st.edge[(size_t)tile * kTileNodes + tid] == tid) {
        uint32_t site;
        (void)node_root_of(st.nodes, tile * kTileNodes + tid, site);
        const u32x4 c = philox(site >> 7, lat.state[0] + t_off, 0u, kTagSwFlip << 28, lat.k0, lat.k1);
        f = (pick4(c, (site >> 5) & 3u) >> (site & 31u)) & 1u;
    }
    flip[tid] = (uint8_t)f;
    __syncthreads();
    // 16 sites a thread: the coins of the runs that start there (site map 0 and
    // its flip are 0 elsewhere)
    uint32_t w = 0;
    const uint32_t d[4] = {ids.x, ids.y, ids.z, ids.w};
#pragma unroll
    for (uint32_t k = 0; k < 16u; ++k) w |= (uint32_t)flip[(d[k >> 2] >> (8u * (k & 3u))) & 0xFFu] << k;
    w <<= 16u * (tid & 1u);
    w |= (uint32_t)__shfl_xor((int)w, 1, 64);
    if (tid & 1u) return;
    const uint32_t i = tid >> 1, tiles_x = L / kTile, tx = tile & (tiles_x - 1u), ty = tile >> ilog2u(tiles_x);
    const uint32_t y = ty * kTile + (i >> 1), x = tx * kTile + 32u * (i & 1u);
    uint32_t *bits = st.bits + y * wpr + (x >> 5);
    const uint32_t s = *bits ^ ((r + w) ^ r);
    *bits = s;
    if (last) sw_store32(lat.spins + (size_t)y * L + x, s);
}

// Level 0 from the bits: operators by words, and level 1 by its words.
__global__ __launch_bounds__(256) void k_sw_measure0(const HbmLattice *__restrict__ lats, uint32_t t_off)
{
    __shared__ uint32_t part[4][4];
    const HbmLattice &lat = lats[blockIdx.y];
    const uint32_t L = (uint32_t)lat.L, i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t *bits = sw_tiles(lat).bits;
    uint32_t c[4] = {0u, 0u, 0u, 0u};
    rm_ops_item(bits, L, i, c[0], c[1], c[2]);
    c[3] = (uint32_t)popc(bits[i]);
    if (i < rm_block_items(L))
        lat.lvl[i] = rm_block_item(bits, L, i, tie_coin_word(i, lat.state[0] + t_off, 0u, lat.k0, lat.k1));
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) {
        c[k] = group_sum(c[k], 64u);
        if ((threadIdx.x & 63u) == 0u) part[k][threadIdx.x >> 6] = c[k];
    }
    __syncthreads();
    if (threadIdx.x < 4u) {
        const uint32_t k = threadIdx.x;
        atomicAdd(lat.sums + k, (unsigned long long)(part[k][0] + part[k][1] + part[k][2] + part[k][3]));
    }
}

size_t sw_scratch_bytes(int L) { return sw_tiles_words((uint32_t)L) * 4u; }

hipError_t launch_sw_sweep(const HbmLattice *d, int n_lats, int L, uint32_t t_off, bool first, bool last, hipStream_t s)
{
    const uint32_t tiles = (uint32_t)((int64_t)L * L / kTileSites);
    const dim3 grid(tiles, (uint32_t)n_lats);
    // few tiles: more threads for each
    if ((int64_t)tiles * n_lats <= 512)
        hipLaunchKernelGGL(k_sw_tile<8>, grid, dim3(kTileSites / 8u), 0, s, d, t_off, first ? 1u : 0u);
    else
        hipLaunchKernelGGL(k_sw_tile<16>, grid, dim3(kTileSites / 16u), 0, s, d, t_off, first ? 1u : 0u);
    hipLaunchKernelGGL(k_sw_seam, dim3(tiles / 2u, (uint32_t)n_lats), dim3(256), 0, s, d);
    hipLaunchKernelGGL(k_sw_apply, grid, dim3(256), 0, s, d, t_off, last ? 1u : 0u);
    return hipGetLastError();
}

hipError_t launch_sw_measure0(const HbmLattice *d, int n_lats, int L, uint32_t t_off, hipStream_t s)
{
    hipLaunchKernelGGL(k_sw_measure0, dim3((uint32_t)((int64_t)L * L / 32 / 256), (uint32_t)n_lats), dim3(256), 0, s, d,
                       t_off);
    return hipGetLastError();
}

}  // namespace mcrg
