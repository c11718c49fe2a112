// indexer_band.hip -- the indexer scores of a fused select (indexer -> top-k) without running
// the exact vector-ALU kernel over every key.
//
// The selection has to be the one the reference makes (src/attention.c:573-598,
// src/ds_model.c:1108-1152): bit-identical scores for every key that could change it.  Most
// keys cannot.  So:
//
//   1. indexer_approx_kernel: approximate scores on the bf16 matrix cores,
//          st[t] = ks[t] * sum_h w[h] * max(q_h . e_t, 0),
//      and next to them a bound on |st[t] - s[t]|, s the reference's score.  The products
//      e*q are exact in fp32 either way (a 4-bit times an 8-bit significand); the two sides
//      differ in the order of the additions and in a handful of roundings:
//          reference dot (dot_f32: four fma chains of 32, three additions)  35 roundings
//          matrix-core dot, any order and any internal truncation          <= 256 roundings
//          scale, weight, sum over at most 64 heads, on each side          <= 2 * 66 roundings
//      each relative to A_h = sum_i |e_i||q_hi| >= |q_h . e_t|, so
//          |st - s| <= 450 u * ks[t] * sum_h |w_h| A_h[t],   u = 2^-24,
//      and sum_h |w_h| A_h[t] = sum_i |e_ti| c_i with c_i = sum_h |w_h||q_hi|: one more row
//      through the matrix core, the key bytes as they are without their signs against c in three E4M3
//      terms, rounded up (at most a 2048th more).  beta[t] = 512 u * ks[t] * that row (the slack covers
//      the rounding of the bound itself: the FP8 matrix core adds up eight products at a time and drops
//      the bits of each below 2^-13 of the largest, a thousandth of the sum at most); beta = max_t beta[t].
//   2. top-k machinery on st: T = the k-th largest approximate score, to the counter it is in: the
//      approximate kernel counts its scores in 4096 of them per row, a 128th of an octave wide in the
//      fourteen octaves where a row's large scores are (topk.hip; band_counter, common.hpp).
//   3. classify: at most k-1 keys have st > T.  A key with st > T + 2 beta has s > T + beta, and
//      every key that scores at least as much has st > T: it is among at most k-2 others, so it
//      is selected whatever the ties do.  At least k keys have st >= T, hence s >= T - beta; a
//      key with st < T - 2 beta has s < T - beta and is not selected.  The first kind gets +inf,
//      the second -inf, the rest (about a hundred of 65536) are candidates.
//   4. indexer_rescore_kernel: the reference's arithmetic, instruction for instruction as in
//      indexer.hip, for the candidates only, spread over heads so that it takes microseconds.
//   5. the selection is the +inf keys (fewer than k, all selected) and the best k - (their number)
//      candidates by exact score, ties to the smaller index: topk_band_finish_kernel (topk.hip)
//      ranks the candidates and writes the indices in order.
// Whenever a row does not fit this (more candidates than the list holds, a bound that is not
// finite, NaN where T should be), the rescoring kernel's workgroups run the exact kernel's code
// on all keys of that row and the finish kernel's first workgroup the plain select.
#include "indexer_exact.hpp"

namespace cwick {

constexpr int IB_THREADS = 512;
constexpr int IB_WAVES = IB_THREADS / 64;
constexpr int IB_QROW = 128 + 8;                 // bf16 per head row of q in LDS (padded: 272 bytes)
constexpr int IB_HD = CWICK_HIP_INDEX_DIM;    // 128

constexpr int IB_TERMS = 3;                      // E4M3 terms of a coefficient of the bound

typedef __attribute__((ext_vector_type(2))) float ib_f32x2;
typedef __attribute__((ext_vector_type(8))) int ib_i32x8;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;

// The (biased) exponent that the bound row's E4M3 coefficients are laid out by, from the largest one's
// bits: kept where 2^(e - 7) and a bound's 512 u times it are normal numbers.
__device__ __forceinline__ uint32_t ib_bound_exponent(uint32_t top) {
    const uint32_t e = top >> 23;
    return e < 24u ? 24u : (e > 254u ? 254u : e);
}

// v[l] + v[l ^ 32] in every lane: the two halves of the wave trade places between two copies
__device__ __forceinline__ float ib_half_sum(float v) {
    float a = v, b = v;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
    return a + b;
}

// What bounds this kernel is the matrix and the vector instructions of an iteration, which two waves
// per SIMD do one after the other.  The bound row on the FP8 matrix core takes 64 cycles per 32 keys (as a
// row of a bf16 product, 31 others of which were zero, 256, and four instructions per k-step to clear
// the signs of the converted keys), and up to 32 heads take one block of them, not one of zeros beside it.
// Sparse decode, 8 rows of 65536 keys 52.0 -> 51.0 us, of 32 heads 50.8 -> 49.3; 4 rows 37.6 -> 35.9.  The rows of
// the product that were free take two more terms of the coefficients: the bound is 5e-5 to 1e-4 above what 64 bits
// give (1024 to 65536 keys, 32 and 64 heads), 4e-2 to 5e-2 with the first term alone and rounded up, 3e-3 with
// coefficients in bf16; 8 rows of 65536 keys 46.7 us with one term and 46.8 with three.
// (The keys of a third iteration in flight: 51.4 and 49.5.)
template <int IB_KEYS, int NB>                  // keys per workgroup, blocks of 32 heads
__global__ void __launch_bounds__(IB_THREADS) __attribute__((amdgpu_waves_per_eu(2)))
indexer_approx_kernel(const uint8_t *__restrict__ keys, const float *__restrict__ kscale,
                      int64_t key_bstride, int64_t kscale_bstride, int64_t n_keys,
                      const uint16_t *__restrict__ q,   // [batch][ih][128] bf16
                      const float *__restrict__ w,      // [batch][ih]
                      int ih, float *__restrict__ scores, float *__restrict__ beta_slots,
                      IndexerBandRow *__restrict__ rows,
                      uint32_t *__restrict__ digits) {   // or null: [batch][slots][CWICK_BAND_DIGITS]
    __shared__ __attribute__((aligned(16))) float cpart_sh[IB_THREADS / 16][IB_HD];
    __shared__ __attribute__((aligned(16))) uint8_t cb_sh[IB_TERMS * IB_HD + 64];    // coefficients' terms, then 64 zeros
    __shared__ __attribute__((aligned(16))) uint32_t counts[4096];
    __shared__ __attribute__((aligned(16))) uint16_t q_sh[64 * IB_QROW];
    __shared__ float w_sh[64];
    __shared__ uint32_t bmax_sh[IB_THREADS / 64];
    __shared__ uint32_t cmax_sh[2];
    const int b = blockIdx.y, wg = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint16_t *qb = q + (size_t)b * ih * IB_HD;
    const float *wb = w + (size_t)b * ih;
    if (wg == 0 && tid == 0) {
        rows[b].n_cand = 0u;
        rows[b].fallback = 0u;
    }
    // Contraction slot j of k-step ks in lane half g is dimension 64 g + 8 ks + j (the same on
    // both operands, so the order is free): a lane reads 64 contiguous bytes of its key row,
    // four 16-byte loads, and a wave reads 32 whole rows.
    const int row = lane & 31, g = lane >> 5;
    const uint8_t *kb = keys + (size_t)b * key_bstride;
    const float *ksb = kscale + (size_t)b * kscale_bstride;
    // (the waves' blocks of 32 keys side by side, 32 KB per turn of the workgroup: a stretch for each wave put all waves
    // of the chip at the same place of a 32 KB piece.  8 rows of 65536 keys of 64 heads again and again 52.3 -> 51.4 us, of
    // 32 49.1 -> 48.5; on keys that the chip's memory cache does not have no difference, 56.4 to 57.7 and 53.3 to 54.8)
    const int64_t wbase = (int64_t)wg * IB_KEYS + wave * 32;
    constexpr int IB_TURN = IB_WAVES * 32, N_IT = IB_KEYS / IB_TURN;
    // the key bytes and the scale of an iteration are loaded two iterations ahead
    u32x4 raw_a[4], raw_b[4], raw_c[4];
    float kst_a, kst_b, kst_c;
    auto load_keys = [&](int it, u32x4 (&raw)[4], float &kst) {
        int64_t tc = wbase + it * IB_TURN + row;
        tc = tc < n_keys ? tc : n_keys - 1;
        const uint8_t *krow = kb + (size_t)tc * IB_HD + 64 * g;
#pragma unroll
        for (int i = 0; i < 4; i++) raw[i] = *(const u32x4 *)(krow + 16 * i);
        kst = ksb[tc];
    };
    // A operands (rows = heads): every wave needs all of q, so the workgroup fetches it once
    // (sixteen bytes per thread and step) and the waves take their fragments from LDS; rows are
    // 272 bytes apart there, which spreads the sixteen-byte reads of consecutive heads over the
    // banks.  The loads go out first and the first two key iterations right behind them.
    // c_i = sum_h |w_h| |q_hi| starts from the same registers: thread (group = tid / 16, part =
    // tid % 16) holds dims 8 part .. +7 of heads group + 16 j, adds up its four heads and leaves
    // the eight sums in LDS; after the barrier thread i < 128 adds the sixteen groups of dim i.
    bf16x8 qa[NB][8];
    // Key scales from four places of the row, the same ones in every workgroup.  (From 64 places, a cache line
    // each in front of the first keys, the kernel takes 0.3 us longer.)
    uint32_t ks_bits;
    {
        // (the weights first: a load that is waited for drags every load issued before it along)
        const float w_mine = (tid < 64 && tid < ih) ? wb[tid] : 0.0f;
        constexpr int NST = 1024 / IB_THREADS;              // sixteen-byte pieces of q per thread
        float w4[NST];
        u32x4 stage[NST];
#pragma unroll
        for (int j = 0; j < NST; j++) {
            const int head = (tid >> 4) + (IB_THREADS / 16) * j;
            w4[j] = head < ih ? fabsf(wb[head]) : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < NST; j++) {
            const int c = tid + IB_THREADS * j, head = c >> 4, part = c & 15;
            const int hc = head < ih ? head : ih - 1;           // clamped load, zeroed afterwards
            stage[j] = *(const u32x4 *)(qb + (size_t)hc * IB_HD + 8 * part);
            if (head >= ih) stage[j] = (u32x4){0u, 0u, 0u, 0u};
        }
        const int64_t ks_at = ((int64_t)(lane >> 4) * n_keys >> 2) + (lane & 15);
        ks_bits = __builtin_bit_cast(uint32_t, ksb[ks_at < n_keys ? ks_at : n_keys - 1]);
        load_keys(0, raw_a, kst_a);
        load_keys(1, raw_b, kst_b);
        float cp[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < NST; j++) {
            const int c = tid + IB_THREADS * j;
            *(u32x4 *)&q_sh[(c >> 4) * IB_QROW + 8 * (c & 15)] = stage[j];
#pragma unroll
            for (int d = 0; d < 4; d++) {
                const uint32_t x = stage[j][d];
                cp[2 * d] = __builtin_fmaf(w4[j], __builtin_bit_cast(float, (x << 16) & 0x7FFFFFFFu), cp[2 * d]);
                cp[2 * d + 1] = __builtin_fmaf(w4[j], __builtin_bit_cast(float, x & 0x7FFF0000u), cp[2 * d + 1]);
            }
        }
        *(f32x4 *)&cpart_sh[tid >> 4][8 * (tid & 15)] = (f32x4){cp[0], cp[1], cp[2], cp[3]};
        *(f32x4 *)&cpart_sh[tid >> 4][8 * (tid & 15) + 4] = (f32x4){cp[4], cp[5], cp[6], cp[7]};
        if (tid < 64) w_sh[tid] = w_mine;
    }
#pragma unroll
    for (int j = 0; j < 4096 / IB_THREADS; j++) counts[tid + IB_THREADS * j] = 0u;
    __syncthreads();
#pragma unroll
    for (int mb = 0; mb < NB; mb++)
#pragma unroll
        for (int ks = 0; ks < 8; ks++)
            qa[mb][ks] = *(const bf16x8 *)&q_sh[(mb * 32 + row) * IB_QROW + 64 * g + 8 * ks];
    float c = 0.0f;                                                                     // never negative
    if (tid < IB_HD) {
        float part[IB_THREADS / 16];
#pragma unroll
        for (int k = 0; k < IB_THREADS / 16; k++) part[k] = cpart_sh[k][tid];
#pragma unroll
        for (int k = 0; k < IB_THREADS / 16; k++) c += part[k];
        const uint32_t top = wave_max_u32(__builtin_bit_cast(uint32_t, c));
        if (lane == 0) cmax_sh[wave] = top;
    }
    __syncthreads();
    const uint32_t c_top = cmax_sh[0] > cmax_sh[1] ? cmax_sh[0] : cmax_sh[1];
    const uint32_t c_exp = ib_bound_exponent(c_top);
    if (tid < IB_HD) {
        // The coefficients over 2^(exponent of the largest - 7), 128 <= largest < 256, in terms of four bits, each
        // a sixteenth of the one before: what is left of one is below 16.  The last is rounded up, what is
        // left below 2^-6, the smallest normal number of E4M3, to that: 2^-21 of the largest coefficient.
        float x = c * __builtin_bit_cast(float, (261u - c_exp) << 23);                  // (NaN: see bound_unit)
#pragma unroll
        for (int t = 0; t < IB_TERMS; t++) {
            uint32_t bits = __builtin_bit_cast(uint32_t, x) & 0xFFF00000u;
            if (t + 1 == IB_TERMS) {
                const float up = x > 0.015625f ? x : 0.015625f;
                bits = x > 0.0f ? __builtin_bit_cast(uint32_t, up) + 0xFFFFFu : 0u;
            }
            cb_sh[IB_HD * t + tid] = bits < 121u << 23 ? 0 : (uint8_t)((bits >> 20) - (120u << 3));
            x = (bits < 121u << 23 ? x : x - __builtin_bit_cast(float, bits)) * 16.0f;
        }
        if (tid < 64) cb_sh[IB_TERMS * IB_HD + tid] = 0;
    }
    // the heads this lane holds after the MFMAs: register i of block mb is head
    // 32 mb + 8 (i / 4) + 4 g + i % 4
    float wl[NB][16];
#pragma unroll
    for (int mb = 0; mb < NB; mb++)
#pragma unroll
        for (int i = 0; i < 16; i++) wl[mb][i] = w_sh[mb * 32 + (i >> 2) * 8 + 4 * g + (i & 3)];

    // The octaves that get most of the counters: a score is at most ks sum_i |e_i| c_i <= ks 448 * 128 max c,
    // so the largest are around 2^16 ks max c, for the ks whose exponent a quarter of the sample reaches
    // (scales of 0 and 1, which keys of zeros have, left out), and what threshold a selection has lies
    // 2 to 13 octaves below that (heads that agree; signed weights that cancel).  Every wave of the row
    // finds the same ones; what they are decides how many candidates there are, not which keys win.  (Here,
    // where the keys are still on their way: each wave for itself, so that no barrier waits for the sample.)
    uint32_t octave;
    {
        const uint32_t e = ks_bits == 0x3F800000u ? 0u : ks_bits >> 23 & 0xFFu;
        const int quarter = (__builtin_popcountll(__ballot(e != 0u)) + 3) / 4;
        uint32_t upper = 0u;
#pragma unroll
        for (int bit = 7; bit >= 0; bit--)
            if (__builtin_popcountll(__ballot(e >= (upper | 1u << bit))) >= quarter) upper |= 1u << bit;
        int lowest = (int)(c_top >> 23 & 0xFFu) + (int)(quarter ? upper : 127u) - 127 + 16 - ((int)BAND_OCTAVES - 1);
        lowest = lowest < 0 ? 0 : lowest;
        lowest = lowest > 256 - (int)BAND_OCTAVES ? 256 - (int)BAND_OCTAVES : lowest;
        octave = (uint32_t)__builtin_amdgcn_readfirstlane(lowest);
    }
    if (wg == 0 && tid == 0) rows[b].octave = octave;
    __syncthreads();                                                // cb_sh

    // The bound row's A fragments.  As operand of a 16x16x128 product a lane's key bytes are column
    // lane % 16, contraction block lane / 16: blocks 0 and 2 hold key `column`, dims 0.. and 64..,
    // blocks 1 and 3 the same dims of key column + 16.  Rows t and 8 + t have term t of the coefficients in blocks
    // 0 and 2, rows 4 + t and 12 + t in blocks 1 and 3, so that register t of every lane is the sum of its own key.
    const int arow = lane & 15, ablk = lane >> 4, term = arow & 3;
    const bool has_c = term < IB_TERMS && ((arow >> 2 ^ ablk) & 1) == 0;
    ib_i32x8 ca[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const lds_u32x4 *src = (const lds_u32x4 *)(const char __attribute__((address_space(3))) *)&cb_sh[
            has_c ? IB_HD * term + 64 * (ablk >> 1) + 32 * h : IB_TERMS * IB_HD + 32 * h];
        const u32x4 lo = src[0], hi = src[1];
        ca[h] = (ib_i32x8){(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
    }
    // 512 u in the coefficients' scale; an infinite or NaN coefficient makes every bound of the row NaN
    const float bound_unit = c_top >= 0x7F800000u ? __builtin_bit_cast(float, 0x7FC00000u)
                                                  : 512.0f / 16777216.0f * __builtin_bit_cast(float, (c_exp - 7u) << 23);

    uint32_t bmax = 0u;      // bits of the largest bound: never negative, they order like the values, NaNs on top
    auto iteration = [&](int it, const u32x4 (&raw)[4], float kst) {
        const int64_t t = wbase + it * IB_TURN + row;
        const bool live = t < n_keys;
        // The accumulators are pinned to VGPRs (through the builtin they land in AGPRs and cost a
        // read each).  The compiler does not see these as MFMAs and leaves out the wait states
        // they need (one state = four cycles = one pass of the matrix pipe): two between a VALU
        // write of an operand and the MFMA that reads it, up to nineteen between the issue of
        // an MFMA and a VALU read of its result.  The first is met by converting the keys
        // of k-step ks + 1 before the MFMAs of k-step ks are issued (which also puts the
        // conversions in the shadow of the matrix pipe), the second by the s_nop behind the loop.
        f32x16 d0, d1;
        // The bound row: a product the compiler knows, in front of the others and read behind them.  Its
        // operands and its result are tied to the assembly below, or it would be moved behind the loop,
        // under the branch of the keys that exist.
        f32x4 ab = {0.0f, 0.0f, 0.0f, 0.0f};
        ib_i32x8 em;
#pragma unroll
        for (int h = 0; h < 2; h++) {
#pragma unroll
            for (int j = 0; j < 8; j++) em[j] = (int)(raw[2 * h + (j >> 2)][j & 3] & 0x7F7F7F7Fu);
            ab = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(ca[h], em, ab, 0, 0, 0, 0x7F7F7F7F, 0, 0x7F7F7F7F);
        }
        __builtin_amdgcn_sched_barrier(0);
        typedef __attribute__((ext_vector_type(2))) __bf16 ib_bf16x2;
        u32x4 e[2];
        auto convert = [&](int ks, u32x4 &eo) {
#pragma unroll
            for (int j = 0; j < 2; j++) {                          // exact: E4M3 fits bf16
                const int dw = raw[ks >> 1][2 * (ks & 1) + j];
                eo[2 * j] = __builtin_bit_cast(uint32_t, (ib_bf16x2)__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(dw, 1.0f, false));
                eo[2 * j + 1] = __builtin_bit_cast(uint32_t, (ib_bf16x2)__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(dw, 1.0f, true));
            }
        };
        convert(0, e[0]);
#pragma unroll
        for (int ks = 0; ks < 8; ks++) {
            const int cur = ks & 1, nxt = cur ^ 1;
            const u32x4 e_before = e[nxt];                          // an operand of the last MFMA issued
            if (ks + 1 < 8) convert(ks + 1, e[nxt]);
            // Everything above is in its registers before the first MFMA below is issued; the
            // operands of the step before stay allocated up to here (an MFMA goes on reading its
            // operands for a while after it has been issued, and the compiler, which does not
            // know, would hand their registers to the conversions above).
            if (ks == 0)
                asm volatile("s_nop 1" : "+v"(e[nxt]), "+v"(e[cur]), "+v"(ab) : "v"(em));
            else
                asm volatile("" : "+v"(e[nxt]), "+v"(e[cur]) : "v"(e_before));
            if (ks == 0) {
                asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(d0) : "v"(qa[0][ks]), "v"(e[cur]));
                if constexpr (NB == 2)
                    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(d1) : "v"(qa[NB - 1][ks]), "v"(e[cur]));
            } else {
                asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d0) : "v"(qa[0][ks]), "v"(e[cur]));
                if constexpr (NB == 2)
                    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d1) : "v"(qa[NB - 1][ks]), "v"(e[cur]));
            }
        }
        // Nothing may read the results or write a register that these MFMAs read before the last
        // one is through: the wait carries the accumulators, so that nothing that reads them can
        // be scheduled above it either.
        if constexpr (NB == 2)
            asm volatile("s_nop 15\n\ts_nop 2" : "+v"(d0), "+v"(d1), "+v"(ab) : "v"(e[1]) : "memory");
        else
            asm volatile("s_nop 15\n\ts_nop 2" : "+v"(d0), "+v"(ab) : "v"(e[1]) : "memory");
        float sp = 0.0f, sq = 0.0f, sr = 0.0f, ss = 0.0f;      // four chains: a dependent FMA waits for the one before it
#pragma unroll
        for (int i = 0; i < 16; i++) {
            // one instruction per ReLU (through fmaxf or fmed3 the compiler adds a second one
            // that quiets NaNs; a NaN dot counts as 0 here, and the bound row turns NaN with it)
            float r0;
            asm("v_max_f32 %0, 0, %1" : "=v"(r0) : "v"(d0[i]));
            if constexpr (NB == 2) {
                float r1;
                asm("v_max_f32 %0, 0, %1" : "=v"(r1) : "v"(d1[i]));
                if (i & 1) {
                    sr = __builtin_fmaf(wl[0][i], r0, sr);
                    ss = __builtin_fmaf(wl[NB - 1][i], r1, ss);
                } else {
                    sp = __builtin_fmaf(wl[0][i], r0, sp);
                    sq = __builtin_fmaf(wl[NB - 1][i], r1, sq);
                }
            } else {
                float &chain = (i & 3) == 0 ? sp : (i & 3) == 1 ? sr : (i & 3) == 2 ? sq : ss;
                chain = __builtin_fmaf(wl[0][i], r0, chain);
            }
        }
        sp = (sp + sq) + (sr + ss);
        // lane l + lane l ^ 32 without a trip through LDS
        sp = ib_half_sum(sp);
        const float st = sp * kst;
        const float band = __builtin_fmaf(ab[2], 1.0f / 256.0f, __builtin_fmaf(ab[1], 1.0f / 16.0f, ab[0]));
        const float beta = band * fabsf(kst) * bound_unit;
        if (live && g == 0) {
            scores[(size_t)b * n_keys + t] = st;
            // the select's pass over the scores, done here
            atomicAdd(&counts[band_counter(st, octave)], 1u);
        }
        const uint32_t bits = __builtin_bit_cast(uint32_t, beta);
        if (live) bmax = bits > bmax ? bits : bmax;
    };
    // three register sets in turn, so that the loads of iteration it + 2 go out before
    // iteration it computes and nothing is copied between sets (a copy waits for its load);
    // unrolled, so that every wait counts exactly the loads behind the one it needs
#pragma unroll
    for (int it = 0; it < N_IT; it += 3) {
        if (wbase + it * IB_TURN >= n_keys) break;                 // wave-uniform
        if (it + 2 < N_IT) load_keys(it + 2, raw_c, kst_c);
        iteration(it, raw_a, kst_a);
        if (it + 1 >= N_IT || wbase + (it + 1) * IB_TURN >= n_keys) break;
        if (it + 3 < N_IT) load_keys(it + 3, raw_a, kst_a);
        iteration(it + 1, raw_b, kst_b);
        if (it + 2 >= N_IT || wbase + (it + 2) * IB_TURN >= n_keys) break;
        if (it + 4 < N_IT) load_keys(it + 4, raw_b, kst_b);
        iteration(it + 2, raw_c, kst_c);
    }
    bmax = wave_max_u32(bmax);
    if (lane == 0) bmax_sh[wave] = bmax;
    __syncthreads();
    if (tid == 0) {
        uint32_t m = bmax_sh[0];
#pragma unroll
        for (int i = 1; i < IB_THREADS / 64; i++) m = bmax_sh[i] > m ? bmax_sh[i] : m;
        beta_slots[(size_t)b * gridDim.x + wg] = __builtin_bit_cast(float, m);
    }
    if (digits && tid < 256) {
        // thread t: counters 16 t .. + 15
        uint32_t *slot = digits + ((size_t)b * gridDim.x + wg) * CWICK_BAND_DIGITS;
        u32x4 c[4];
#pragma unroll
        for (int j = 0; j < 4; j++) c[j] = *(const u32x4 *)&counts[16 * tid + 4 * j];
        u32x4 w[2];
#pragma unroll
        for (int j = 0; j < 8; j++) w[j >> 2][j & 3] = c[j >> 1][2 * (j & 1)] | c[j >> 1][2 * (j & 1) + 1] << 16;   // at most 2048 each
        const u32x4 s4 = (c[0] + c[1]) + (c[2] + c[3]);
        slot[tid] = (s4[0] + s4[1]) + (s4[2] + s4[3]);
        *(u32x4 *)&slot[256 + 8 * tid] = w[0];
        *(u32x4 *)&slot[256 + 8 * tid + 4] = w[1];
    }
}

// The reference's score of each candidate, written over its approximate one.  One workgroup
// = 16 candidates x 16 groups of four heads: lane j of a row of sixteen lanes holds candidate
// j's key, the row its four heads; the dot products run exactly as in indexer_scores_kernel
// (the q values of a head come to the FMAs through DPP row broadcasts); the 64 weighted terms
// of a candidate meet in LDS and one lane adds them in head order.
__global__ void __launch_bounds__(256)
indexer_rescore_kernel(const int32_t *__restrict__ cand, const IndexerBandRow *__restrict__ rows, int n_keys32, int cap,
                       const uint16_t *__restrict__ q, const float *__restrict__ w, int ih,
                       // (up to here they arrive in registers)
                       const uint8_t *__restrict__ keys, const float *__restrict__ kscale,
                       int64_t key_bstride, int64_t kscale_bstride, float *__restrict__ scores,
                       float *__restrict__ cand_score) {   // [batch][cap]: the same scores in list order
    __shared__ __attribute__((aligned(16))) float terms[16][68];
    const int b = blockIdx.y, tid = threadIdx.x;
    const int64_t n_keys = n_keys32;
    int c0 = blockIdx.x * 16;
    const int j = tid & 15, hg = tid >> 4;                          // candidate, head group
    // The list entry is fetched next to the row's state, not behind it (one round trip less in
    // front of the key's bytes): an entry past the end of the list is whatever the workspace
    // held, so it is clamped to a key of the row; what is computed for it is not stored.
    int64_t t_guess = cand[(size_t)b * cap + c0 + j];
    // q of the group's four heads, on its way beside them: lane j holds q[h][8 j .. 8 j + 7]
    const uint16_t *qb = q + (size_t)b * ih * IB_HD;
    const float *wb = w + (size_t)b * ih;
    u32x4 qraw[4];
    float wh[4];
#pragma unroll
    for (int hh = 0; hh < 4; hh++) {
        const int h = hg * 4 + hh;
        const int hc = h < ih ? h : ih - 1;
        qraw[hh] = *(const u32x4 *)(qb + (size_t)hc * IB_HD + 8 * j);
        wh[hh] = wb[hc];
    }
    IndexerBandRow st;                                              // the two words in use, not the padding
    st.n_cand = rows[b].n_cand;
    st.fallback = rows[b].fallback;
    t_guess = t_guess < 0 ? 0 : (t_guess >= n_keys ? n_keys - 1 : t_guess);
    if (indexer_band_failed(st, cap)) {
        // the row did not fit the band: the workgroups of this launch score all of its keys
        // with the exact kernel's code instead
        for (int64_t block = blockIdx.x; block * IDX_THREADS < n_keys; block += gridDim.x) {
            indexer_exact_block(keys, kscale, key_bstride, kscale_bstride, n_keys, q, w, ih, scores, b, block);
            __syncthreads();
        }
        return;
    }
    // a list longer than the launch covers in one go (rare) takes further rounds
    for (; c0 < (int)st.n_cand; c0 += (int)gridDim.x * 16) {
    int64_t t = t_guess;                                            // (a slot past the end scores some key of the row: not stored)
    if (c0 != (int)blockIdx.x * 16) {
        t = cand[(size_t)b * cap + c0 + j];
        t = t < 0 ? 0 : (t >= n_keys ? n_keys - 1 : t);
    }
    const uint8_t *krow = keys + (size_t)b * key_bstride + (size_t)t * IB_HD;
    const float ks = kscale[(size_t)b * kscale_bstride + t];
    float e[IB_HD];
#pragma unroll
    for (int c = 0; c < IB_HD / 16; c++) {
        const u32x4 v = *(const u32x4 *)(krow + c * 16);
#pragma unroll
        for (int jj = 0; jj < 4; jj++) {
            const f32x2 lo = e4m3x2_to_f32<false>(v[jj]);
            const f32x2 hi = e4m3x2_to_f32<true>(v[jj]);
            e[c * 16 + jj * 4 + 0] = lo[0];
            e[c * 16 + jj * 4 + 1] = lo[1];
            e[c * 16 + jj * 4 + 2] = hi[0];
            e[c * 16 + jj * 4 + 3] = hi[1];
        }
    }
    f32x4 mine;
#pragma unroll
    for (int hh = 0; hh < 4; hh++) {
        const int h = hg * 4 + hh;
        float qv[8];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            qv[2 * c] = bf16lo_to_f32(qraw[hh][c]);
            qv[2 * c + 1] = bf16hi_to_f32(qraw[hh][c]);
        }
        // the loaded values pass through an (empty) VALU instruction: what the DPP reads below
        // is then ordinary data to the compiler, which sees to the waits; the two wait states a
        // DPP read needs after a VALU write are spent in the accumulator initialisation
#pragma unroll
        for (int c = 0; c < 8; c++) asm volatile("" : "+v"(qv[c]));
        float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
        asm volatile("s_nop 1" ::: "memory");
#define CWICK_IB_FMA(acc, n, c)                                                                    \
    asm volatile("v_fmac_f32_dpp %0, %1, %2 row_newbcast:" #n " row_mask:0xf bank_mask:0xf"       \
                 : "+v"(acc) : "v"(qv[c]), "v"(e[8 * n + c]))
#define CWICK_IB_EIGHT(n)                                                                          \
    CWICK_IB_FMA(s0, n, 0); CWICK_IB_FMA(s1, n, 1); CWICK_IB_FMA(s2, n, 2); CWICK_IB_FMA(s3, n, 3);   \
    CWICK_IB_FMA(s0, n, 4); CWICK_IB_FMA(s1, n, 5); CWICK_IB_FMA(s2, n, 6); CWICK_IB_FMA(s3, n, 7)
        CWICK_IB_EIGHT(0); CWICK_IB_EIGHT(1); CWICK_IB_EIGHT(2); CWICK_IB_EIGHT(3);
        CWICK_IB_EIGHT(4); CWICK_IB_EIGHT(5); CWICK_IB_EIGHT(6); CWICK_IB_EIGHT(7);
        CWICK_IB_EIGHT(8); CWICK_IB_EIGHT(9); CWICK_IB_EIGHT(10); CWICK_IB_EIGHT(11);
        CWICK_IB_EIGHT(12); CWICK_IB_EIGHT(13); CWICK_IB_EIGHT(14); CWICK_IB_EIGHT(15);
#undef CWICK_IB_EIGHT
#undef CWICK_IB_FMA
        float d = (s0 + s1) + (s2 + s3);
        d = d * ks;
        d = d < 0.0f ? 0.0f : d;
        const float prod = d * wh[hh];
        mine[hh] = h < ih ? prod : 0.0f;
    }
    *(f32x4 *)&terms[j][4 * hg] = mine;
    __syncthreads();
    if (tid < 16 && c0 + tid < (int)st.n_cand) {
        f32x4 x[16];                                                // (all terms at once; past the last head a zero)
#pragma unroll
        for (int h = 0; h < 16; h++) x[h] = *(const f32x4 *)&terms[tid][4 * h];
        float s = 0.0f;
#pragma unroll
        for (int h = 0; h < 64; h++) s = s + x[h >> 2][h & 3];
        scores[(size_t)b * n_keys + t] = s;                         // (candidate j is thread j's own)
        cand_score[(size_t)b * cap + c0 + tid] = s;
    }
    __syncthreads();                                                // before the next round's terms
    }
}

template <int NB>
static auto indexer_approx_of(int per) {
    return per == 512 ? indexer_approx_kernel<512, NB> : per == 768 ? indexer_approx_kernel<768, NB> :
           per == 1024 ? indexer_approx_kernel<1024, NB> : per == 1536 ? indexer_approx_kernel<1536, NB> :
           indexer_approx_kernel<CWICK_INDEXER_APPROX_KEYS, NB>;
}

// the approximate scores and the per-workgroup maxima of their error bound (the first stage of
// the banded select on its own; n_keys / IB_KEYS slots per row, rounded up)
int launch_indexer_approx(const uint8_t *keys, const float *kscale, int64_t key_bstride,
                          int64_t kscale_bstride, int batch, int64_t n_keys, const uint16_t *q_idx,
                          const float *w, int n_idx_heads, float *scores, float *beta_slots,
                          IndexerBandRow *rows, uint32_t *digits, hipStream_t s) {
    static_assert(IB_THREADS >= 256 && 1024 % IB_THREADS == 0, "a thread per first-digit bin, whole pieces of q per thread");
    CWICK_REQUIRE(keys && kscale && q_idx && w && scores && beta_slots && rows, "indexer_approx: null pointer");
    CWICK_REQUIRE(n_keys >= 1 && n_idx_heads >= 1 && n_idx_heads <= 64, "indexer_approx: shape out of range");
    CWICK_REQUIRE((uintptr_t)keys % 16 == 0 && key_bstride % 16 == 0 && (uintptr_t)q_idx % 16 == 0,
                  "indexer_approx: keys and q must be 16-byte aligned");
    const int n_wg = indexer_approx_slots(n_keys, batch), per = indexer_approx_keys(n_keys, batch);
    {
        ProfKernel pk(CWICK_HIP_PROF_INDEXER_APPROX, s);
        const auto kernel = n_idx_heads > 32 ? indexer_approx_of<2>(per) : indexer_approx_of<1>(per);
        pk.launch(kernel, dim3(n_wg, batch), dim3(IB_THREADS), 0, keys, kscale, key_bstride, kscale_bstride,
                  n_keys, q_idx, w, n_idx_heads, scores, beta_slots, rows, digits);
    }
    CWICK_HIP_CALL(hipGetLastError());
    return 1;
}

int launch_indexer_banded(const uint8_t *keys, const float *kscale, int64_t key_bstride,
                          int64_t kscale_bstride, int batch, int64_t n_keys, const uint16_t *q_idx,
                          const float *w, int n_idx_heads, int64_t k, float *scores, int32_t *out_idx,
                          hipStream_t s) {
    CWICK_REQUIRE(keys && kscale && q_idx && w && scores && out_idx, "indexer_banded: null pointer");
    CWICK_REQUIRE(indexer_band_applies(n_keys, k, n_idx_heads, batch), "indexer_banded: shape out of range");
    CWICK_REQUIRE((uintptr_t)keys % 16 == 0 && key_bstride % 16 == 0 && (uintptr_t)q_idx % 16 == 0,
                  "indexer_banded: keys and q must be 16-byte aligned");
    const int n_wg = indexer_approx_slots(n_keys, batch);
    constexpr int cap = CWICK_INDEXER_BAND_CAP;
    // workspace: [digit counts][beta slots][row states][+inf counts][candidate lists][their exact scores]
    const size_t digit_bytes = indexer_band_digits_dwords(n_keys, batch) * sizeof(uint32_t);
    size_t off_beta = (digit_bytes + 255) & ~(size_t)255;
    size_t off_rows = off_beta + (((size_t)batch * n_wg * sizeof(float) + 255) & ~(size_t)255);
    size_t off_hi = off_rows + (((size_t)batch * sizeof(IndexerBandRow) + 255) & ~(size_t)255);
    size_t off_cand = off_hi + (size_t)batch * 64 * sizeof(uint32_t);
    size_t off_cs = off_cand + (size_t)batch * cap * sizeof(int32_t);
    const size_t total = off_cs + (size_t)batch * cap * sizeof(float);
    char *ws = (char *)workspace(s, total);
    if (!ws) return 0;                      // workspace() has recorded why
    float *beta_slots = (float *)(ws + off_beta);
    IndexerBandRow *rows = (IndexerBandRow *)(ws + off_rows);
    uint32_t *hi_count = (uint32_t *)(ws + off_hi);
    int32_t *cand = (int32_t *)(ws + off_cand);
    float *cand_score = (float *)(ws + off_cs);
    {
    ProfScope ps(CWICK_HIP_PROF_INDEXER, s);
    if (!launch_indexer_approx(keys, kscale, key_bstride, kscale_bstride, batch, n_keys, q_idx, w, n_idx_heads,
                               scores, beta_slots, rows, (uint32_t *)ws, s))
        return 0;
    if (!launch_topk_band_classify(scores, batch, n_keys, k, (const uint32_t *)ws, beta_slots, n_wg, cand, cap, rows,
                                   hi_count, s))
        return 0;
    // Sixteen candidates per workgroup and round, one or two hundred per row: 32 workgroups a row take them in
    // one (8 rows of 64K keys: 56.4 us the step with 8 per row, 53.3 with 16 or 32, 54.6 with 64 or 96; with
    // equal weights 60.3, 56.9, 53.7, 54.9).  With few rows there are more, for a row that scores all of its
    // keys; with many rows fewer, because workgroups that find nothing to do cost their launch.
    int rescore_wgs = num_cus() / batch;
    rescore_wgs = rescore_wgs < 8 ? 8 : (rescore_wgs > cap / 16 ? cap / 16 : rescore_wgs);
    indexer_rescore_kernel<<<dim3(rescore_wgs, batch), 256, 0, s>>>(
        cand, rows, (int)n_keys, cap, q_idx, w, n_idx_heads, keys, kscale, key_bstride, kscale_bstride, scores, cand_score);
    CWICK_HIP_CALL(hipGetLastError());
    }
    return launch_topk_band_finish(scores, batch, n_keys, k, cand, cand_score, cap, rows, hi_count, out_idx, s);
}

}  // namespace cwick
