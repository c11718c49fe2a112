// Block selection of the block-sparse GQA decode (the MiniMax family of the reference).
//
// Replaces, for one query or a chunk of consecutive ones, mm_index_scores (src/mm_model.c:
// 1764-1780), mm_select_blocks (:1733-1761) and the loop that writes the chosen blocks out as
// positions (:1969-1976).  What leaves is a position list per query, padded with -1, that
// launch_gqa_decode takes as its `sel`: the whole selection stays on the device.
//
//   1. mm_index_scores_kernel   one thread per (position, index head): the dot of the head's fp32
//      query with the position's bf16 key, a fused multiply-add per dimension in dimension order
//      from zero (the reference's serial loop: a chain belongs to one thread, but the heads of a
//      position are independent chains), then ReLU and the heads added in head order by the
//      first wave.  A workgroup is 64 positions x one wave per head; a wave's query is uniform
//      and read through the scalar unit; a thread requests its whole 256-byte key row in
//      16-byte pieces before it uses the first.  (mm_index_scores128_kernel: keys of 128 dimensions,
//      one thread per position.)
//   2. block maxima, started from -1e30 like the reference.  The scoring kernel leaves the
//      maximum of every group of 64 positions; when a block is a whole number of groups (128 in
//      the reference's configuration) mm_pick_few_kernel (up to 2048 blocks, 32 kept) or
//      mm_pick_kernel, one workgroup per query, makes the block maxima from them, selects the
//      `keep` best blocks (the radix select in the second, lowest index first among equal maxima --
//      the reference's heap makes that choice on tie-free input) and writes the list: one launch.  Other block sizes take mm_blockmax_kernel (one
//      wave per block over the scores; blocks past a query's last one get -inf so that rows of
//      a chunk with different block counts share one top-k launch), launch_topk and
//      mm_expand_kernel.
//   3. the list: block limit / block is added when it is not among the chosen (for a limit that
//      is a multiple of the block size this is a block without a written position, which
//      contributes nothing -- the reference's rule, kept as it is); chosen blocks are full
//      except the last, so position p of the list is block[p / block] * block + p % block, or
//      -1 past the limit.
#include "common.hpp"
#include "topk_row.hpp"

namespace cwick {
namespace {

constexpr int MM_THREADS = 256;
constexpr int MM_SCORE_THREADS = 64;        // positions per workgroup of the scoring kernel (one wave per index head)
constexpr int MM_MAX_HEADS = 8;
constexpr int64_t MM_SHORT_POSITIONS = 32768;   // up to here the scoring kernel takes a wave per head
constexpr int MM_MAX_DIM = 512;

__global__ void __launch_bounds__(MM_SCORE_THREADS * MM_MAX_HEADS)
mm_index_scores_kernel(const uint16_t *__restrict__ keys, const float *__restrict__ iq, int64_t limit0, int ih, int id,
                       float *__restrict__ scores, int64_t score_stride,
                       float *__restrict__ gmax, int64_t gmax_stride) {
    // workgroup = 64 positions x ih waves: wave h runs head h's chain for the 64 positions (the
    // heads are independent until the sum), its lanes the positions
    __shared__ float sh_d[MM_MAX_HEADS][MM_SCORE_THREADS];
    const int row = blockIdx.y;
    const int64_t limit = limit0 + row;
    if ((int64_t)blockIdx.x * MM_SCORE_THREADS >= limit) return;          // the whole workgroup: before the barrier
    const int lane = threadIdx.x & 63;
    const int h = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t s = (int64_t)blockIdx.x * MM_SCORE_THREADS + lane;
    const int64_t sc = s < limit ? s : limit - 1;                   // threads past the end read the last row
    const u32x4 *kp = (const u32x4 *)(keys + (size_t)sc * id);
    const int chunks = id / 8;
    // sixteen pieces of the row (a whole 128-dimension key) are requested before the first is
    // used: one round trip to memory per key
    constexpr int G = 16;
    u32x4 kw[G];
#pragma unroll
    for (int g = 0; g < G; g++) kw[g] = kp[g < chunks ? g : chunks - 1];
    // the head's query is the same for every lane of the wave: its address is uniform, so it
    // arrives through the scalar unit, eight values a load, and enters the multiply-adds as a
    // scalar operand
    const float *__restrict__ q = iq + ((size_t)row * ih + h) * id;
    float d = 0.0f;
    for (int c0 = 0; c0 < chunks; c0 += G) {
        if (c0) {
#pragma unroll
            for (int g = 0; g < G; g++) kw[g] = kp[c0 + g < chunks ? c0 + g : chunks - 1];
        }
#pragma unroll
        for (int g = 0; g < G; g++) {
            if (c0 + g < chunks) {                                  // uniform
                const float *qc = q + (c0 + g) * 8;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    d = __builtin_fmaf(qc[2 * i], bf16lo_to_f32(kw[g][i]), d);
                    d = __builtin_fmaf(qc[2 * i + 1], bf16hi_to_f32(kw[g][i]), d);
                }
            }
        }
    }
    sh_d[h][lane] = d;
    __syncthreads();
    if (h != 0) return;
    float tot = 0.0f;
    for (int j = 0; j < ih; j++) {
        const float dj = sh_d[j][lane];
        if (dj > 0.0f) tot = tot + dj;
    }
    if (s < limit) scores[(size_t)row * score_stride + s] = tot;
    // the largest score of this group of 64 positions: what the block maxima are made of when a
    // block is a whole number of groups
    if (gmax) {
        const float gm = wave_max(s < limit ? fmaxf(-1e30f, tot) : -INFINITY);
        if ((threadIdx.x & 63) == 0) gmax[(size_t)row * gmax_stride + blockIdx.x] = gm;
    }
}

// The same for long contexts: one thread per position runs the chains of all heads (a key row is
// read by one wave instead of one per head, which is what counts once the rows come from HBM
// rather than out of a cache that the head waves share).
__global__ void __launch_bounds__(MM_SCORE_THREADS)
mm_index_scores_long_kernel(const uint16_t *__restrict__ keys, const float *__restrict__ iq, int64_t limit0, int ih, int id,
                       float *__restrict__ scores, int64_t score_stride,
                       float *__restrict__ gmax, int64_t gmax_stride) {
    const int row = blockIdx.y;
    const int64_t limit = limit0 + row;
    if ((int64_t)blockIdx.x * MM_SCORE_THREADS >= limit) return;
    const int64_t s = (int64_t)blockIdx.x * MM_SCORE_THREADS + threadIdx.x;
    const int64_t sc = s < limit ? s : limit - 1;                   // threads past the end read the last row
    const u32x4 *kp = (const u32x4 *)(keys + (size_t)sc * id);
    const int chunks = id / 8;
    // sixteen pieces of the row (a whole 128-dimension key) are requested before the first is
    // used: one round trip to memory per key
    constexpr int G = 16;
    u32x4 kw[G];
#pragma unroll
    for (int g = 0; g < G; g++) kw[g] = kp[g < chunks ? g : chunks - 1];
    // the query is the same for every thread: its address is uniform, so it arrives through the
    // scalar unit, eight values a load, and enters the multiply-adds as a scalar operand
    const float *__restrict__ q = iq + (size_t)row * ih * id;
    float d[MM_MAX_HEADS];
#pragma unroll
    for (int h = 0; h < MM_MAX_HEADS; h++) d[h] = 0.0f;
    for (int c0 = 0; c0 < chunks; c0 += G) {
        if (c0) {
#pragma unroll
            for (int g = 0; g < G; g++) kw[g] = kp[c0 + g < chunks ? c0 + g : chunks - 1];
        }
#pragma unroll
        for (int g = 0; g < G; g++) {
            if (c0 + g < chunks) {                                  // uniform
                const int c = c0 + g;
                float kf[8];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    kf[2 * i] = bf16lo_to_f32(kw[g][i]);
                    kf[2 * i + 1] = bf16hi_to_f32(kw[g][i]);
                }
#pragma unroll
                for (int h = 0; h < MM_MAX_HEADS; h++) {
                    if (h < ih) {                                   // uniform
                        const float *qh = q + h * id + c * 8;
#pragma unroll
                        for (int i = 0; i < 8; i++) d[h] = __builtin_fmaf(qh[i], kf[i], d[h]);
                    }
                }
            }
        }
    }
    float tot = 0.0f;
#pragma unroll
    for (int h = 0; h < MM_MAX_HEADS; h++)
        if (h < ih && d[h] > 0.0f) tot = tot + d[h];
    if (s < limit) scores[(size_t)row * score_stride + s] = tot;
    // the largest score of this group of 64 positions: what the block maxima are made of when a
    // block is a whole number of groups
    if (gmax) {
        const float gm = wave_max(s < limit ? fmaxf(-1e30f, tot) : -INFINITY);
        if ((threadIdx.x & 63) == 0) gmax[(size_t)row * gmax_stride + blockIdx.x] = gm;
    }
}

// Keys of 128 dimensions: a thread per position runs the chains of all heads, and the queries reach the
// multiply-adds through the vector registers: lane n of each row of sixteen holds q[h][8 n .. 8 n + 7], and
// dimension i is taken from lane i / 8 of register i % 8 by a DPP row broadcast inside the multiply-add.
// (Through the scalar unit every eight dimensions waited for a load: 65536 positions, four heads, 9.7 us of
// which the multiply-adds are 1.3.)  The order of a chain is the same.
template <int IH>
__global__ void __launch_bounds__(MM_SCORE_THREADS)
mm_index_scores128_kernel(const uint16_t *__restrict__ keys, const float *__restrict__ iq, int64_t limit0, int ih,
                          float *__restrict__ scores, int64_t score_stride,
                          float *__restrict__ gmax, int64_t gmax_stride) {
    const int row = blockIdx.y;
    const int64_t limit = limit0 + row;
    if ((int64_t)blockIdx.x * MM_SCORE_THREADS >= limit) return;
    const int lane = threadIdx.x;
    const int64_t s = (int64_t)blockIdx.x * MM_SCORE_THREADS + lane;
    const u32x4 *kp = (const u32x4 *)(keys + (size_t)(s < limit ? s : limit - 1) * 128);    // threads past the end read the last row
    const float *qp = iq + (size_t)row * ih * 128 + 8 * (lane & 15);
    f32x4 q[IH][2];
    u32x4 kw[16];
#pragma unroll
    for (int h = 0; h < IH; h++) {
        const float *qh = qp + (h < ih ? h : ih - 1) * 128;
        q[h][0] = *(const f32x4 *)qh;
        q[h][1] = *(const f32x4 *)(qh + 4);
    }
#pragma unroll
    for (int g = 0; g < 16; g++) kw[g] = kp[g];
    float d[IH];
#pragma unroll
    for (int h = 0; h < IH; h++) d[h] = 0.0f;
    // the queries are in their registers here; the two wait states that a DPP read needs behind a vector
    // write are spent below
#pragma unroll
    for (int h = 0; h < IH; h++) asm volatile("" : "+v"(q[h][0]), "+v"(q[h][1]));
    asm volatile("s_nop 1" ::: "memory");
#define CWICK_MM_FMA(n, i)                                                                            \
    _Pragma("unroll") for (int h = 0; h < IH; h++)                                                     \
        asm volatile("v_fmac_f32_dpp %0, %1, %2 row_newbcast:" #n " row_mask:0xf bank_mask:0xf"        \
                     : "+v"(d[h]) : "v"(q[h][(i) >> 2][(i) & 3]), "v"(kf[i]))
#define CWICK_MM_EIGHT(n)                                                                             \
    do {                                                                                              \
        float kf[8];                                                                                  \
        _Pragma("unroll") for (int i = 0; i < 4; i++) {                                                \
            kf[2 * i] = bf16lo_to_f32(kw[n][i]);                                                      \
            kf[2 * i + 1] = bf16hi_to_f32(kw[n][i]);                                                  \
        }                                                                                             \
        CWICK_MM_FMA(n, 0); CWICK_MM_FMA(n, 1); CWICK_MM_FMA(n, 2); CWICK_MM_FMA(n, 3);               \
        CWICK_MM_FMA(n, 4); CWICK_MM_FMA(n, 5); CWICK_MM_FMA(n, 6); CWICK_MM_FMA(n, 7);               \
    } while (0)
    CWICK_MM_EIGHT(0); CWICK_MM_EIGHT(1); CWICK_MM_EIGHT(2); CWICK_MM_EIGHT(3);
    CWICK_MM_EIGHT(4); CWICK_MM_EIGHT(5); CWICK_MM_EIGHT(6); CWICK_MM_EIGHT(7);
    CWICK_MM_EIGHT(8); CWICK_MM_EIGHT(9); CWICK_MM_EIGHT(10); CWICK_MM_EIGHT(11);
    CWICK_MM_EIGHT(12); CWICK_MM_EIGHT(13); CWICK_MM_EIGHT(14); CWICK_MM_EIGHT(15);
#undef CWICK_MM_EIGHT
#undef CWICK_MM_FMA
    float tot = 0.0f;
#pragma unroll
    for (int h = 0; h < IH; h++)
        if (h < ih && d[h] > 0.0f) tot = tot + d[h];
    if (s < limit) scores[(size_t)row * score_stride + s] = tot;
    if (gmax) {
        const float gm = wave_max(s < limit ? fmaxf(-1e30f, tot) : -INFINITY);
        if (lane == 0) gmax[(size_t)row * gmax_stride + blockIdx.x] = gm;
    }
}

__global__ void __launch_bounds__(MM_THREADS)
mm_blockmax_kernel(const float *__restrict__ scores, int64_t score_stride, int64_t limit0, int bs, int64_t nblk_max,
                   float *__restrict__ bsc) {
    const int lane = threadIdx.x & 63;
    const int64_t b = (int64_t)blockIdx.x * (MM_THREADS / 64) + (threadIdx.x >> 6);
    const int row = blockIdx.y;
    if (b >= nblk_max) return;
    const int64_t limit = limit0 + row;
    const int64_t lo = b * bs, hi = lo + bs < limit ? lo + bs : limit;
    float mx = lo < limit ? -1e30f : -INFINITY;
    const float *sc = scores + (size_t)row * score_stride;
    for (int64_t t = lo + lane; t < hi; t += 64) mx = fmaxf(mx, sc[t]);
    mx = wave_max(mx);
    if (lane == 0) bsc[(size_t)row * nblk_max + b] = mx;
}

// The list of one query, by all NT threads of a workgroup: the first `nv` of `mine` are the chosen blocks in
// ascending order, the newest block among them (`has`) or not.
template <int NT>
__device__ __forceinline__ void mm_write_row(const int32_t *__restrict__ mine, int nv, bool has, int kb, int64_t limit, int bs,
                                             int32_t *__restrict__ blk_out, int32_t *__restrict__ sel, int64_t max_sel,
                                             int32_t *__restrict__ n_sel) {
    const int tid = threadIdx.x;
    const int32_t newest = (int32_t)(limit / bs);
    const int nb = nv + (has ? 0 : 1);
    if (blk_out)
        for (int j = tid; j <= kb; j += NT) blk_out[j] = j < nv ? mine[j] : j < nb ? newest : -1;
    // every block of the list but its last is full
    for (int64_t p = tid; p < max_sel; p += NT) {
        const int64_t j = (uint32_t)p / (uint32_t)bs;                 // (both fit: a 64-bit division is a hundred instructions)
        int64_t pos = -1;
        if (j < nb) {
            const int64_t b = j < nv ? mine[j] : newest;
            pos = b * bs + (p - j * bs);
            if (pos >= limit) pos = -1;
        }
        sel[p] = (int32_t)pos;
    }
    if (n_sel && tid == 0) {
        const int64_t last = nb - 1 < nv ? mine[nb - 1] : newest;
        int64_t in_last = limit - last * bs;
        in_last = in_last < 0 ? 0 : in_last > bs ? bs : in_last;
        const int64_t total = (int64_t)(nb - 1) * bs + in_last;
        *n_sel = (int32_t)(total < max_sel ? total : max_sel);
    }
}

// The same where `mine` holds kb chosen blocks in ascending order, -1 padded.
template <int NT>
__device__ __forceinline__ void mm_expand_row(const int32_t *__restrict__ mine, int kb, int64_t limit, int bs,
                                              int32_t *__restrict__ blk_out, int32_t *__restrict__ sel, int64_t max_sel,
                                              int32_t *__restrict__ n_sel) {
    __shared__ uint32_t sh_nv, sh_has;
    const int tid = threadIdx.x;
    const int64_t nblk = (limit + bs - 1) / bs;
    const int32_t newest = (int32_t)(limit / bs);
    if (tid == 0) sh_nv = 0, sh_has = 0;
    __syncthreads();
    // the chosen blocks come in ascending order, blocks this query does not have (and the -1
    // padding of a short row) after the ones it has: the valid entries are a prefix
    for (int j0 = 0; j0 < kb; j0 += NT) {
        const int j = j0 + tid;
        const int32_t b = j < kb ? mine[j] : -1;
        const uint32_t ok = b >= 0 && b < nblk;
        const uint32_t cnt = wave_sum_u32(ok), has = wave_sum_u32(ok && b == newest);
        if ((tid & 63) == 0 && cnt) atomicAdd(&sh_nv, cnt);
        if ((tid & 63) == 0 && has) atomicAdd(&sh_has, has);
    }
    __syncthreads();
    mm_write_row<NT>(mine, (int)sh_nv, sh_has != 0u, kb, limit, bs, blk_out, sel, max_sel, n_sel);
}

__global__ void __launch_bounds__(MM_THREADS)
mm_expand_kernel(const int32_t *__restrict__ blk, int kb, int64_t limit0, int bs, int32_t *__restrict__ blk_out,
                 int32_t *__restrict__ sel, int64_t max_sel, int32_t *__restrict__ n_sel) {
    const int row = blockIdx.x;
    mm_expand_row<MM_THREADS>(blk + (size_t)row * kb, kb, limit0 + row, bs,
                              blk_out ? blk_out + (size_t)row * (kb + 1) : nullptr, sel + (size_t)row * max_sel, max_sel,
                              n_sel ? n_sel + row : nullptr);
}

// Block maxima, the kept blocks and the list of one query in one workgroup, for up to 2048 blocks that are a whole
// number of the scoring kernel's 64-position groups, of which at most 32 are kept.
//
// Nothing here but the trip to the group maxima takes long by itself, so what counts is the chain: the radix select
// has ten barriers of sixteen waves between that trip and the list, this four of eight.  The kk-th largest of 64
// maxima, each of every 64th block, is a bound that kk blocks reach and few others do (32 of them: some 44), found bit
// by bit from counts of ballots, by every wave for itself.  Where the blocks that reach it are at most 64 they go
// into a lane each of the first wave, in order, which finds the threshold in the same way, until as many as are wanted
// reach it.  65536 positions in blocks of 128, sixteen kept: 5.2 us by the radix select, 3.5; 131072 in blocks of 64: 5.8,
// 3.6.  (The first wave alone with a lane for every 64th block: 4.1 and 8.2.)
//
// Where more blocks reach it, by ties or because the largest share lanes, the whole workgroup counts, three bits of
// the threshold to a barrier.  The whole selection of 16 of 2048 blocks, us, by the radix select and so: all
// equal 19.9 and 11.1, eight levels 15.5 and 11.1, a hundred equal above the rest 15.3 and 14.7, four in one lane
// of every wave 13.5 and 12.9, distinct 13.7 and 10.9; of 512 blocks 13.4 and 9.2, 12.4 and 9.2, 12.6 and 9.2, 12.4 and
// 9.3, 11.4 and 9.5.  (The first wave alone, bit by bit, all equal: 63 and 22.6.)
//
// More than 32 are kept by the radix select: the 36th largest of 64 maxima has 53 blocks above it on the average
// and the 64th nearly all, so that counting is what is left.  64 of 2048 distinct blocks 14.3 us by the radix select and
// 17.8 by counts of the workgroup, of 512 blocks 12.3 and 13.3.
constexpr int MM_PICK_THREADS = 512, MM_PICK_WAVES = MM_PICK_THREADS / 64, MM_PICK_KEEP = 32, MM_PICK_BLOCKS = 2048;
template <int EPT>
__global__ void __launch_bounds__(MM_PICK_THREADS)
mm_pick_few_kernel(const float *__restrict__ gmax, int64_t gmax_stride, int64_t limit0, int bs, int kb,
                   int32_t *__restrict__ blk_out, int32_t *__restrict__ sel, int64_t max_sel, int32_t *__restrict__ n_sel) {
    __shared__ uint32_t sh_top[MM_PICK_WAVES][64], sh_cand[64], sh_of[MM_PICK_WAVES][2];
    __shared__ __attribute__((aligned(16))) uint32_t sh_digit[2][MM_PICK_WAVES][4];
    __shared__ int32_t sh_idx[64], sh_blk[MM_PICK_KEEP];
    __shared__ uint32_t sh_cnt[MM_PICK_WAVES], sh_has;
    const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int limit = (int)(limit0 + row);
    const int nblk = (limit + bs - 1) / bs, ngrp = (limit + 63) / 64, gpb = bs / 64;
    const int kk = kb < nblk ? kb : nblk, newest = limit / bs;
    const float *gm = gmax + (size_t)row * gmax_stride;
    // element j of this lane is block first + 64 j
    const int first = wave * (64 * EPT) + lane;
    float v[EPT];
#pragma unroll
    for (int j = 0; j < EPT; j++) v[j] = -1e30f;
    for (int u = 0; u < gpb; u += 4)                                    // four groups of each block at a time
#pragma unroll
        for (int j = 0; j < EPT; j++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int b = first + 64 * j < nblk ? first + 64 * j : nblk - 1;     // (past the end: the last block's)
                const int g = b * gpb + (u + i < gpb ? u + i : gpb - 1);
                v[j] = fmaxf(v[j], gm[g < ngrp ? g : ngrp - 1]);
            }
    uint32_t key[EPT], top = 0u;                                        // (no block's key is 0)
#pragma unroll
    for (int j = 0; j < EPT; j++) {
        key[j] = first + 64 * j < nblk ? topk_key(v[j]) : 0u;
        top = key[j] > top ? key[j] : top;
    }
    sh_top[wave][lane] = top;
    if (tid == 0) sh_has = 0u;
    __syncthreads();
    auto count = [](bool x) { return __builtin_popcountll(__ballot(x)); };
    auto below = [](uint64_t m) {                                       // lanes below this one in m
        return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
    };
    // the largest T that at least kk of what `reach` counts reach, or the first found that exactly kk do (`all`)
    auto threshold = [&](auto reach, bool &all) {
        uint32_t T = 0u;
        all = false;
        for (uint32_t bit = 0x80000000u; bit; bit >>= 1) {
            const int c = reach(T | bit);
            if (c >= kk) T |= bit;
            if (c == kk) {
                all = true;
                break;
            }
        }
        return T;
    };
    bool all;
#pragma unroll
    for (int w = 0; w < MM_PICK_WAVES; w++) top = sh_top[w][lane] > top ? sh_top[w][lane] : top;
    const uint32_t bound = threshold([&](uint32_t x) { return count(top >= x); }, all);
    uint64_t in[EPT];
    int n_in = 0;
#pragma unroll
    for (int j = 0; j < EPT; j++) {
        in[j] = __ballot(key[j] >= bound && key[j]);
        n_in += __builtin_popcountll(in[j]);
    }
    if (lane == 0) sh_cnt[wave] = (uint32_t)n_in;
    __syncthreads();
    int at = 0, n_cand = 0;
#pragma unroll
    for (int w = 0; w < MM_PICK_WAVES; w++) {
        if (w < wave) at += (int)sh_cnt[w];
        n_cand += (int)sh_cnt[w];
    }
    if (n_cand <= 64) {                                                 // uniform
#pragma unroll
        for (int j = 0; j < EPT; j++) {
            if (in[j] >> lane & 1) {
                sh_cand[at + below(in[j])] = key[j];
                sh_idx[at + below(in[j])] = first + 64 * j;
            }
            at += __builtin_popcountll(in[j]);
        }
        __syncthreads();
    }
    if (n_cand <= 64) {
        if (wave == 0) {
            const uint32_t mine = lane < n_cand ? sh_cand[lane] : 0u;
            const uint32_t T = threshold([&](uint32_t x) { return count(mine >= x); }, all);
            // ties at T that do not all fit: the smaller indices win
            const int r = kk - count(mine > T);
            const bool tied = mine == T && mine, take = mine && (all ? mine >= T : mine > T || (tied && below(__ballot(tied)) < r));
            const uint64_t m = __ballot(take);
            bool has = false;
            if (take) {
                const int idx = sh_idx[lane];
                sh_blk[below(m)] = idx;
                has = idx == newest;
            }
            const uint64_t any = __ballot(has);
            if (lane == 0) sh_has = any != 0u;
        }
    } else {
        // Three bits at a time, from the first in which the bound and the largest maximum differ (equal scores: none at
        // all).  Every lane counts its blocks by digit, a nibble each; what is added up over the workgroup
        // are the blocks up to each digit, digits d and d + 4 in the halves of word d.
        const uint32_t most = wave_max_u32(top);
        int bits = bound == most ? 0 : 32 - __builtin_clz(bound ^ most);
        uint32_t T = bits == 32 ? 0u : bound >> bits << bits;
        for (int turn = 0; bits > 0; turn ^= 1) {
            const int shift = bits > 3 ? bits - 3 : 0;                  // (fewer bits left: no block reaches the values past them)
            uint32_t seen = 0u;
#pragma unroll
            for (int j = 0; j < EPT; j++) {
                const uint32_t d = (key[j] - T) >> shift;
                seen += 1u << 4 * (key[j] < T ? 0u : d < 7u ? d : 7u);
            }
            seen *= 0x11111111u;
            u32x4 up_to;
#pragma unroll
            for (int d = 0; d < 4; d++) up_to[d] = wave_sum_u32(seen >> 4 * d & 0x000F000Fu);
            if (lane == 0) *(u32x4 *)sh_digit[turn][wave] = up_to;
            __syncthreads();
            uint32_t sum = 0u;                                          // for lanes 1 .. 7: blocks below the value of this digit
#pragma unroll
            for (int w = 0; w < MM_PICK_WAVES; w++) sum += sh_digit[turn][w][(lane - 1) & 3];
            const int reach = MM_PICK_THREADS * EPT - (int)(lane > 4 ? sum >> 16 : sum & 0xFFFFu);
            const int digit = count(lane > 0 && lane < 8 && reach >= kk);       // (more blocks reach the smaller values)
            T += (uint32_t)digit << shift;
            bits = digit && __builtin_amdgcn_readlane(reach, digit) == kk ? 0 : shift;
        }
        int over = 0, ties = 0;                                         // of this wave
        uint64_t m_eq[EPT];
#pragma unroll
        for (int j = 0; j < EPT; j++) {
            over += count(key[j] > T);
            m_eq[j] = __ballot(key[j] == T);
            ties += __builtin_popcountll(m_eq[j]);
        }
        if (lane == 0) sh_of[wave][0] = (uint32_t)over, sh_of[wave][1] = (uint32_t)ties;
        __syncthreads();
        int r = kk, to = 0, tied = 0;                                   // ties that are selected; places and ties in front of this wave
#pragma unroll
        for (int w = 0; w < MM_PICK_WAVES; w++) {
            const int o = (int)sh_of[w][0], e = (int)sh_of[w][1];
            r -= o;
            if (w < wave) to += o, tied += e;
        }
        to += tied < r ? tied : r;
#pragma unroll
        for (int j = 0; j < EPT; j++) {
            const bool take = key[j] > T || (key[j] == T && tied + below(m_eq[j]) < r);
            const uint64_t m = __ballot(take);
            if (take) {
                sh_blk[to + below(m)] = first + 64 * j;
                if (first + 64 * j == newest) sh_has = 1u;
            }
            to += __builtin_popcountll(m);
            tied += __builtin_popcountll(m_eq[j]);
        }
    }
    __syncthreads();
    mm_write_row<MM_PICK_THREADS>(sh_blk, kk, sh_has != 0u, kb, limit, bs, blk_out ? blk_out + (size_t)row * (kb + 1) : nullptr,
                                  sel + (size_t)row * max_sel, max_sel, n_sel ? n_sel + row : nullptr);
}

// The same for any number of blocks, of which any number is kept: blocks that are
// a whole number of the scoring kernel's 64-position groups: a block's maximum is that of its
// groups (a few KB per query instead of the scores themselves), the selection is the
// one-workgroup radix select, the list follows.  Three launches less than the general path.
__global__ void __launch_bounds__(TOPK_THREADS)
mm_pick_kernel(const float *__restrict__ gmax, int64_t gmax_stride, int64_t limit0, int bs, int64_t nblk_max, int kb,
               float *__restrict__ bsc, int32_t *__restrict__ blk, int32_t *__restrict__ blk_out,
               int32_t *__restrict__ sel, int64_t max_sel, int32_t *__restrict__ n_sel) {
    const int row = blockIdx.x, tid = threadIdx.x;
    const int64_t limit = limit0 + row;
    const int64_t nblk = (limit + bs - 1) / bs, ngrp = (limit + 63) / 64;
    const int gpb = bs / 64;                                          // groups per block
    const float *gm = gmax + (size_t)row * gmax_stride;
    auto block_max = [&](int64_t b) {
        float mx = -1e30f;
        for (int u = 0; u < gpb; u++) {
            const int64_t gi = b * gpb + u;
            if (gi < ngrp) mx = fmaxf(mx, gm[gi]);
        }
        return mx;
    };
    int32_t *out_blk = blk_out ? blk_out + (size_t)row * (kb + 1) : nullptr, *out_sel = sel + (size_t)row * max_sel;
    int32_t *out_n = n_sel ? n_sel + row : nullptr;
    if (nblk <= 4 * TOPK_THREADS && kb <= TOPK_THREADS) {
        // what the steps hand on stays in LDS: through memory every hand-over is a round trip
        __shared__ float sh_bsc[4 * TOPK_THREADS];
        __shared__ int32_t sh_blk[TOPK_THREADS];
        for (int64_t b = tid; b < nblk; b += TOPK_THREADS) sh_bsc[b] = block_max(b);
        __syncthreads();
        if (nblk <= TOPK_THREADS) topk_radix_reg_row<1>(sh_bsc, nblk, kb, sh_blk);     // a score per thread, kept in a register
        else topk_radix_reg_row<4>(sh_bsc, nblk, kb, sh_blk);
        __syncthreads();
        mm_expand_row<TOPK_THREADS>(sh_blk, kb, limit, bs, out_blk, out_sel, max_sel, out_n);
        return;
    }
    float *mybsc = bsc + (size_t)row * nblk_max;
    for (int64_t b = tid; b < nblk; b += TOPK_THREADS) mybsc[b] = block_max(b);
    __syncthreads();                                                  // the workgroup reads what it wrote
    int32_t *myblk = blk + (size_t)row * kb;
    topk_radix_row(mybsc, nblk, kb, myblk);
    __syncthreads();
    mm_expand_row<TOPK_THREADS>(myblk, kb, limit, bs, out_blk, out_sel, max_sel, out_n);
}

}  // namespace

int launch_mm_select(const uint16_t *idx_keys, const float *iq, int batch, int64_t limit0, int index_heads,
                     int index_dim, int block, int keep_blocks, float *scores, int64_t score_stride,
                     int32_t *blk_out, int32_t *sel, int64_t max_sel, int32_t *n_sel, hipStream_t s) {
    CWICK_REQUIRE(idx_keys && iq && scores && sel, "mm_select: null pointer");
    CWICK_REQUIRE(batch >= 1 && batch <= 65535 && limit0 >= 1 && limit0 + batch - 1 <= ((int64_t)1 << 30),
                  "mm_select: batch %d, first limit %lld", batch, (long long)limit0);
    CWICK_REQUIRE(index_heads >= 1 && index_heads <= MM_MAX_HEADS && index_dim >= 8 && index_dim <= MM_MAX_DIM &&
                      index_dim % 8 == 0,
                  "mm_select: %d index heads of %d dims (1..%d heads, dims a multiple of 8 up to %d)", index_heads,
                  index_dim, MM_MAX_HEADS, MM_MAX_DIM);
    CWICK_REQUIRE(block >= 1 && keep_blocks >= 1 && keep_blocks <= 4096, "mm_select: block %d, blocks kept %d", block,
                  keep_blocks);
    const int64_t limit_max = limit0 + batch - 1;
    CWICK_REQUIRE(score_stride >= limit_max, "mm_select: score rows of %lld hold fewer than %lld positions",
                  (long long)score_stride, (long long)limit_max);
    CWICK_REQUIRE(max_sel >= 1 && max_sel <= ((int64_t)1 << 24), "mm_select: max_sel %lld", (long long)max_sel);
    CWICK_REQUIRE(((uintptr_t)idx_keys) % 16 == 0, "mm_select: index keys must be 16-byte aligned");
    const int64_t nblk_max = (limit_max + block - 1) / block;
    // (the top-k below keeps its own workspace slot, so the block scores can sit in this call's)
    CWICK_REQUIRE(nblk_max < 16384, "mm_select: %lld blocks (at most 16383)", (long long)nblk_max);
    const bool fused = block % MM_SCORE_THREADS == 0;          // a block is whole groups of the scoring kernel
    const int64_t ng_max = (limit_max + MM_SCORE_THREADS - 1) / MM_SCORE_THREADS;
    const size_t bsc_b = ((size_t)batch * nblk_max * 4 + 255) & ~(size_t)255;
    const size_t blk_b = ((size_t)batch * keep_blocks * 4 + 255) & ~(size_t)255;
    char *ws = (char *)workspace(s, bsc_b + blk_b + (fused ? (size_t)batch * ng_max * 4 : 0));
    if (!ws) return 0;                      // workspace() has recorded why
    float *bsc = (float *)ws;
    int32_t *blk = (int32_t *)(ws + bsc_b);
    float *gmax = fused ? (float *)(ws + bsc_b + blk_b) : nullptr;
    {
        ProfScope ps(CWICK_HIP_PROF_MM_SELECT, s);
        const dim3 sgrid((unsigned)ng_max, batch);
        // up to 32 K positions a wave per head (8 192 positions: 8.5 -> 5.5 us); beyond, the head
        // waves' reads of the same key rows cost more than their parallelism gains (262 144
        // positions: 19 us against 32)
        if (index_dim == 128 && (uintptr_t)iq % 16 == 0) {
            auto scores128 = index_heads == 1 ? mm_index_scores128_kernel<1>
                             : index_heads == 2 ? mm_index_scores128_kernel<2>
                             : index_heads <= 4 ? mm_index_scores128_kernel<4> : mm_index_scores128_kernel<8>;
            scores128<<<sgrid, MM_SCORE_THREADS, 0, s>>>(idx_keys, iq, limit0, index_heads, scores, score_stride, gmax, ng_max);
        } else if (limit_max * batch <= MM_SHORT_POSITIONS)
            mm_index_scores_kernel<<<sgrid, MM_SCORE_THREADS * index_heads, 0, s>>>(
                idx_keys, iq, limit0, index_heads, index_dim, scores, score_stride, gmax, ng_max);
        else
            mm_index_scores_long_kernel<<<sgrid, MM_SCORE_THREADS, 0, s>>>(idx_keys, iq, limit0, index_heads, index_dim,
                                                                       scores, score_stride, gmax, ng_max);
        if (fused && nblk_max <= MM_PICK_BLOCKS && keep_blocks <= MM_PICK_KEEP)
            (nblk_max <= MM_PICK_THREADS ? mm_pick_few_kernel<1> : mm_pick_few_kernel<MM_PICK_BLOCKS / MM_PICK_THREADS>)<<<dim3(batch), MM_PICK_THREADS, 0, s>>>(
                gmax, ng_max, limit0, block, keep_blocks, blk_out, sel, max_sel, n_sel);
        else if (fused)
            mm_pick_kernel<<<dim3(batch), TOPK_THREADS, 0, s>>>(gmax, ng_max, limit0, block, nblk_max, keep_blocks, bsc,
                                                                blk, blk_out, sel, max_sel, n_sel);
        else
            mm_blockmax_kernel<<<dim3((unsigned)((nblk_max + 3) / 4), batch), MM_THREADS, 0, s>>>(
                scores, score_stride, limit0, block, nblk_max, bsc);
    }
    CWICK_HIP_CALL(hipGetLastError());
    if (fused) return 1;
    if (!launch_topk(bsc, batch, nblk_max, keep_blocks, blk, s)) return 0;
    {
        ProfScope ps(CWICK_HIP_PROF_MM_SELECT, s);
        mm_expand_kernel<<<dim3(batch), MM_THREADS, 0, s>>>(blk, keep_blocks, limit0, block, blk_out, sel, max_sel, n_sel);
    }
    CWICK_HIP_CALL(hipGetLastError());
    return 1;
}

}  // namespace cwick
