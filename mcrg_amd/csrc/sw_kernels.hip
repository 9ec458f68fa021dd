// Swendsen-Wang cluster sweeps: the Wolff construction (src/ising.cpp:96-149)
// for every cluster at once, with union-find on bit-packed bonds (sw_core.hpp).
//
//   k_sw_wg   a whole lattice of L <= kSwWgMaxL in one workgroup's LDS, for all
//             the sweeps of a launch, with the measurement of every level and
//             the records (src/lattice.cpp:102-120, src/mcrg.cpp:72-98, :314-348)
#include <algorithm>
#include <mutex>

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
    static std::mutex mu;
    static uint32_t opted_in = 65536u;
    {
        std::lock_guard<std::mutex> lk(mu);
        if (lds_bytes > opted_in) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_sw_wg<PW>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
            if (e != hipSuccess) return e;
            opted_in = lds_bytes;
        }
    }
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
    uint32_t lds_bytes = 4u * sw_wg_layout((uint32_t)L, (uint32_t)n_levels, n_work).total;
    // No more workgroups on one compute unit than an even share: LDS is asked
    // for that keeps the others out, or some units would take six and others
    // two (1024 lattices of L = 64).
    const uint32_t share = (uint32_t)((n_lats + n_cus - 1) / n_cus);
    if (share <= 8u) lds_bytes = std::max(lds_bytes, kMaxLdsBytes / share / 2048u * 2048u);
    switch (part) {
    case 4: return launch_sw_wg_pw<4>(d, n_lats, lds_bytes, n, measure, n_work, threads, s);
    case 8: return launch_sw_wg_pw<8>(d, n_lats, lds_bytes, n, measure, n_work, threads, s);
    case 16: return launch_sw_wg_pw<16>(d, n_lats, lds_bytes, n, measure, n_work, threads, s);
    case 32: return launch_sw_wg_pw<32>(d, n_lats, lds_bytes, n, measure, n_work, threads, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace mcrg
