// topk_row.hpp -- the radix select of one row by one workgroup of TOPK_THREADS threads, shared by
// the top-k kernels (topk.hip) and by kernels that select inside a larger step (mm_select.hip).
// Order: (score descending, index ascending); the k best are written in ascending index order;
// entries past min(k, n) are filled with -1.
#pragma once
#include "common.hpp"

#include <type_traits>

namespace cwick {

constexpr int TOPK_THREADS = 1024;
constexpr int TOPK_WAVES = TOPK_THREADS / 64;

// exclusive scan of one value per thread across the block; returns the
// exclusive prefix and writes the block total to *total
__device__ __forceinline__ uint32_t block_exscan(uint32_t v, uint32_t *sh_wave, uint32_t *total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t inc = wave_scan_u32(v);
    if (lane == 63) sh_wave[wave] = inc;
    __syncthreads();
    uint32_t wave_off = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < TOPK_WAVES; w++) {
        const uint32_t c = sh_wave[w];
        if (w < wave) wave_off += c;
        tot += c;
    }
    __syncthreads();
    *total = tot;
    return wave_off + inc - v;
}

// one row by one workgroup of TOPK_THREADS; sc and dst are the row's
__device__ __forceinline__ void topk_radix_row(const float *__restrict__ sc, int64_t n, int64_t k,
                                               int32_t *__restrict__ dst) {
    // 16 copies of the histogram, picked by lane, so that the lanes of a wave
    // that hit one digit (scores cluster in a few exponent buckets) do not all
    // serialise on one LDS word
    __shared__ uint32_t hist16[256 * 16];
    __shared__ uint32_t hist[256];
    __shared__ uint32_t sh_wave[TOPK_WAVES];
    __shared__ uint32_t sh_prefix, sh_remaining;
    const int tid = threadIdx.x;
    const int64_t kk = k < n ? k : n;

    for (int64_t i = kk + tid; i < k; i += TOPK_THREADS) dst[i] = -1;

    if (tid == 0) {
        sh_prefix = 0u;
        sh_remaining = (uint32_t)kk;
    }
    // ---- 1. find the key of the kk-th best element ----
    uint32_t prefix = 0u, mask = 0u;
    for (int shift = 24; shift >= 0; shift -= 8) {
#pragma unroll
        for (int j = 0; j < 4; j++) hist16[tid * 4 + j] = 0u;
        __syncthreads();
        for (int64_t i = tid; i < n; i += TOPK_THREADS) {
            const uint32_t key = topk_key(sc[i]);
            if ((key & mask) == prefix)
                atomicAdd(&hist16[((key >> shift) & 0xFFu) * 16 + (tid & 15)], 1u);
        }
        __syncthreads();
        if (tid < 256) {
            uint32_t c = 0u;
#pragma unroll
            for (int j = 0; j < 16; j++) c += hist16[tid * 16 + j];
            hist[tid] = c;
        }
        __syncthreads();
        if (tid < 64) {
            // walk the 256 buckets from the largest digit down; lane b owns
            // buckets 255-4b .. 252-4b
            const uint32_t remaining = sh_remaining;
            uint32_t c[4], sum = 0u;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                c[j] = hist[255 - (tid * 4 + j)];
                sum += c[j];
            }
            uint32_t inc = wave_scan_u32(sum);
            uint32_t before = inc - sum;   // elements in strictly larger buckets
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (before < remaining && remaining <= before + c[j]) {
                    sh_prefix = prefix | ((uint32_t)(255 - (tid * 4 + j)) << shift);
                    sh_remaining = remaining - before;
                }
                before += c[j];
            }
        }
        __syncthreads();
        prefix = sh_prefix;
        mask |= 0xFFu << shift;
    }
    const uint32_t T = prefix;
    const uint32_t r = sh_remaining;   // elements equal to T that belong to the selection

    // ---- 2. ordered emit ----
    uint32_t out_base = 0u, eq_base = 0u;
    for (int64_t base = 0; base < n; base += (int64_t)TOPK_THREADS * 4) {
        const int64_t i0 = base + (int64_t)tid * 4;
        uint32_t key[4];
#pragma unroll
        for (int j = 0; j < 4; j++) key[j] = (i0 + j < n) ? topk_key(sc[i0 + j]) : 0u;
        uint32_t n_eq = 0u;
#pragma unroll
        for (int j = 0; j < 4; j++) n_eq += (i0 + j < n && key[j] == T) ? 1u : 0u;
        uint32_t eq_total;
        uint32_t eq_before = eq_base + block_exscan(n_eq, sh_wave, &eq_total);
        uint32_t take[4], n_take = 0u;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const bool in = i0 + j < n;
            const bool gt = in && key[j] > T;
            const bool eq = in && key[j] == T;
            take[j] = (gt || (eq && eq_before < r)) ? 1u : 0u;
            if (eq) eq_before++;
            n_take += take[j];
        }
        uint32_t take_total;
        uint32_t pos = out_base + block_exscan(n_take, sh_wave, &take_total);
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (take[j]) dst[pos++] = (int32_t)(i0 + j);
        out_base += take_total;
        eq_base += eq_total;
    }
}

// ---- rows that fit the register file: n <= TOPK_THREADS * EPT ----
// Wave w owns the consecutive elements [w * 64 * ept, (w + 1) * 64 * ept); inside it lane l
// holds elements base + 64 j + l, so the loads are coalesced and index order is (j, lane):
// positions inside a wave come from ballots, positions of the waves from one scan.
//
// The threshold comes from digits of twelve, twelve and eight bits: 4096 buckets spread the scores of one
// exponent, so that the lanes of a wave rarely meet in one counter, and the passes end as soon as all of
// a bucket belongs to the selection, which after two is nearly always.
//
// One workgroup on one compute unit: what it takes is the vector instructions of its sixteen waves, one after
// the other on each SIMD, and its barriers.  So no comparison with the row's end except in the waves that hold
// it, keys in four instructions, and the search for the bucket left to the wave that has it.  512 of 9001
// positions and the attention over them 27.1 -> 24.0 us, 2048 of 20000 38.9 -> 33.5.  (Eight waves: 25.7 and 37.1;
// four: 31.2 and 58.1.)
#define CWICK_TOPK_EACH(j) _Pragma("unroll") for (int j = 0; j < EPT; j++)
template <int EPT>
__device__ __forceinline__ void topk_radix_reg_row(const float *__restrict__ sc, int64_t n, int64_t k,
                                                   int32_t *__restrict__ dst) {
    constexpr int THREADS = TOPK_THREADS, BINS = 4096, OWN = BINS / THREADS, WAVES = TOPK_WAVES;
    static_assert(OWN % 4 == 0 && WAVES <= 64, "counters in sixteen-byte pieces, a lane per wave");
    __shared__ __attribute__((aligned(16))) uint32_t hist[2][BINS];
    __shared__ __attribute__((aligned(16))) u32x4 sh_pick;
    __shared__ uint32_t sh_sum[WAVES], sh_gt[WAVES], sh_eq[WAVES];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t kk = k < n ? k : n;
    for (int64_t i = kk + tid; i < k; i += THREADS) dst[i] = -1;

    const int ept = (int)((n + THREADS - 1) / THREADS);               // <= EPT
    const int wbase = wave * 64 * ept;
    const bool full = (int64_t)wbase + 64 * ept <= n;                 // no element of the wave is past the end
    // this lane holds elements j < jv
    const int left = (int)n - wbase - lane;
    const int jv = left <= 0 ? 0 : (left + 63) / 64 < ept ? (left + 63) / 64 : ept;
    typedef std::true_type whole;
    typedef std::false_type ends;
    auto mine = [&](auto w, int j) { return decltype(w)::value ? j < ept : j < jv; };     // (the first: the same for the wave)
    uint32_t key[EPT];
    auto read = [&](auto w) {
        const float *p = sc + wbase;
        float v[EPT];
        CWICK_TOPK_EACH(j) v[j] = mine(w, j) ? p[64 * j + lane] : 0.0f;
        CWICK_TOPK_EACH(j) key[j] = topk_key(v[j]);
    };
#pragma unroll
    for (int i = 0; i < OWN; i += 4) {
        *(u32x4 *)&hist[0][4 * tid + THREADS * i] = (u32x4){0u, 0u, 0u, 0u};
        *(u32x4 *)&hist[1][4 * tid + THREADS * i] = (u32x4){0u, 0u, 0u, 0u};
    }
    if (full) read(whole{});
    else read(ends{});
    __syncthreads();
    // ---- 1. the chosen digits of the kk-th best element's key ----
    uint32_t T = 0u, mask = 0u, r = (uint32_t)kk, count = 0u;         // r: how many of the `count` keys with (key & mask) == T are selected
#pragma unroll
    for (int pass = 0; pass < 3; pass++) {
        const int shift = pass == 0 ? 20 : pass == 1 ? 8 : 0;
        const uint32_t low = pass == 2 ? 0xFFu : 0xFFFu;
        uint32_t *h = hist[pass & 1];
        auto tally = [&](auto w) {
            CWICK_TOPK_EACH(j)
                if (mine(w, j) && (pass == 0 || (key[j] & mask) == T)) atomicAdd(&h[key[j] >> shift & low], 1u);
        };
        if (full) tally(whole{});
        else tally(ends{});
        __syncthreads();
        // thread t owns the buckets from BINS - OWN (t + 1) on, so a scan goes from the largest digit down
        u32x4 c[OWN / 4], s4 = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int i = 0; i < OWN / 4; i++) {
            c[i] = *(const u32x4 *)&h[BINS - OWN * (tid + 1) + 4 * i];
            s4 += c[i];
        }
        const uint32_t sum = (s4[0] + s4[1]) + (s4[2] + s4[3]), inc = wave_scan_u32(sum);
        if (lane == 63) sh_sum[wave] = inc;
        if (pass == 0)                                                // for the third pass
#pragma unroll
            for (int i = 0; i < OWN / 4; i++) *(u32x4 *)&h[BINS - OWN * (tid + 1) + 4 * i] = (u32x4){0u, 0u, 0u, 0u};
        __syncthreads();
        const uint32_t of_wave = lane < WAVES ? sh_sum[lane] : 0u;
        const uint32_t larger = (uint32_t)__builtin_amdgcn_readlane((int)(wave_scan_u32(of_wave) - of_wave), wave);
        const uint32_t here = (uint32_t)__builtin_amdgcn_readlane((int)of_wave, wave);
        if (larger < r && r <= larger + here) {                       // uniform: the wave that has the bucket
            uint32_t before = larger + inc - sum;
            if (before < r && r <= before + sum)
#pragma unroll
                for (int i = OWN - 1; i >= 0; i--) {
                    const uint32_t x = c[i >> 2][i & 3];
                    if (before < r && r <= before + x) sh_pick = (u32x4){(uint32_t)(BINS - OWN * (tid + 1) + i), r - before, x, 0u};
                    before += x;
                }
        }
        __syncthreads();
        const u32x4 pick = sh_pick;
        T |= (uint32_t)__builtin_amdgcn_readfirstlane((int)pick[0]) << shift;
        r = (uint32_t)__builtin_amdgcn_readfirstlane((int)pick[1]);
        count = (uint32_t)__builtin_amdgcn_readfirstlane((int)pick[2]);
        mask |= low << shift;
        if (count == r) break;                                        // uniform
    }

    // ---- 2. ordered emit ----
    // what lanes below this one have of m, on top of `pos`
    auto place = [](uint64_t m, uint32_t pos) {
        return (uint32_t)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, pos));
    };
    auto put = [&](uint32_t pos, int j) { *(int32_t *)((char *)dst + (uint32_t)(4 * pos)) = wbase + 64 * j + lane; };
    if (count == r) {
        // everything from T up (the bits of T behind the mask are zero): one ballot per element
        auto total = [&](auto w) {
            uint32_t t = 0u;
            CWICK_TOPK_EACH(j) t += (uint32_t)__builtin_popcountll(__ballot(mine(w, j) && key[j] >= T));
            return t;
        };
        const uint32_t mine_of = full ? total(whole{}) : total(ends{});
        if (lane == 0) sh_gt[wave] = mine_of;
        __syncthreads();
        const uint32_t of_wave = lane < WAVES ? sh_gt[lane] : 0u;
        uint32_t pos = (uint32_t)__builtin_amdgcn_readlane((int)(wave_scan_u32(of_wave) - of_wave), wave);
        auto emit = [&](auto w) {
            CWICK_TOPK_EACH(j) {
                const bool take = mine(w, j) && key[j] >= T;
                const uint64_t m = __ballot(take);
                if (take) put(place(m, pos), j);
                pos += (uint32_t)__builtin_popcountll(m);
            }
        };
        if (full) emit(whole{});
        else emit(ends{});
        return;
    }
    // ties that do not all fit (T is a whole key here): the smaller indices win
    uint32_t w_gt = 0u, w_eq = 0u;         // wave totals (uniform)
    CWICK_TOPK_EACH(j) {
        w_gt += (uint32_t)__builtin_popcountll(__ballot(j < jv && key[j] > T));
        w_eq += (uint32_t)__builtin_popcountll(__ballot(j < jv && key[j] == T));
    }
    if (lane == 0) {
        sh_gt[wave] = w_gt;
        sh_eq[wave] = w_eq;
    }
    __syncthreads();
    uint32_t eq_before = 0u, pos = 0u;     // ties / outputs of the waves before this one
    for (int w = 0; w < wave; w++) {
        const uint32_t e = sh_eq[w];
        const uint32_t take_e = eq_before >= r ? 0u : (r - eq_before < e ? r - eq_before : e);
        pos += sh_gt[w] + take_e;
        eq_before += e;
    }
    CWICK_TOPK_EACH(j) {
        const bool gt = j < jv && key[j] > T;
        const bool eq = j < jv && key[j] == T;
        const uint64_t m_eq = __ballot(eq);
        const bool take = gt || (eq && place(m_eq, eq_before) < r);
        const uint64_t m_take = __ballot(take);
        if (take) put(place(m_take, pos), j);
        pos += (uint32_t)__builtin_popcountll(m_take);
        eq_before += (uint32_t)__builtin_popcountll(m_eq);
    }
}
#undef CWICK_TOPK_EACH

}  // namespace cwick
