// gqa_decode.hip -- split-K flash-decoding for one query position over a bf16
// K/V cache (the decode branch of the reference's mixer_attn,
// src/q35_model.c:1656-1701: dec_scores / dec_softmax / dec_out_slices).
//
// HBM-bound: every K and V row is read exactly once, and nothing but the loads may be in the way.
//
//   grid  = (n_splits, n_kv_heads), 256 threads (4 waves)
//   A workgroup owns one kv head and every n_splits-th step of 64 keys and serves the `group` query
//   heads that share the kv head (the reference walks cache rows for the same reason: one row
//   serves every head of its group, src/q35_model.c:1417-1423).  A wave takes tiles of 16 keys.
//   At any time the workgroups read neighbouring steps, which lie in all channels of the memory.
//   (A contiguous slice each: where its length is a multiple of a power of two, the slices are in the same
//   channels at the same time.  64 heads on 8 x 128, a call on the caches of one layer after the other, some 6 GB of
//   them: 65536 keys 58.0 us, 50.3 so; 131072 103.3 and 94.7; 100003 76.2 and 70.3; 33000 29.9 and 28.9; on the same
//   caches again 57.1, 50.5; 103.0, 95.3; 77.8, 73.9; 29.1, 28.5.  Alone behind 512 MB written to other memory, 100003
//   142 and 137.  The one place where it is the slower: alone on caches that were written whole just before, so that
//   what the chip's memory cache still has is read in another order, 109.5 and 114.)
//
//   scores:  S[key][head] = K Q^T, v_mfma_f32_16x16x32_bf16 straight from registers: lane l reads
//            16 bytes of key l%16 per load, which is the A operand as it lies in the cache.  The
//            16 columns are the query heads (those past the group are zero).
//   values:  O[head][dim] += P V in fp32 (V widened, the weights never rounded).  Lane l of the score
//            result holds head l%16 and keys 4(l/16) .. +4, and reads 16 bytes of the V rows of the
//            same keys: its weights and its values are operands of one matrix product as they are,
//            neither moves between lanes and V takes no trip through LDS.
//            Up to four heads (v_mfma_f32_4x4x1_16b_f32, QUADS = 1): a lane's weight is row l%4 of
//            its block of four lanes (the score columns repeat the heads), its value a column; every
//            lane group keeps the sums of its own keys and the four meet at the end.  8 cycles per
//            64 values; eight heads of 128 dims take two of them (QUADS = 2).
//            More heads (v_mfma_f32_16x16x4_f32, QUADS = 0): register r of the score result is the A
//            operand of a product over the keys {r, 4+r, 8+r, 12+r}.  32 cycles per 64 values: 1100
//            cycles of one SIMD's matrix pipe per 8 KiB tile, a third of what HBM takes for it.
//   (Dots and sums on the vector ALU, a row spread over 16 or 32 lanes, took 194 us for 100003
//   keys of 8 kv heads x 128, eight query heads each: 410 MB at 2.1 TB/s.)
//   softmax: a lane keeps its own part of the weight sum.  The reference of a head is the maximum of
//            the wave's first tile and stays there while later scores exceed it by less than 2^64;
//            a wave that meets a larger score moves it and rescales (rare).
//   The next tile's loads are in flight while a tile is worked on.  The waves of a workgroup meet in
//   LDS, then (m, l, acc) goes to the workspace.  Up to GQA_DEC_LAST_MERGE splits are merged by the last
//   workgroup of the kv head to draw a ticket: the partials are written through and read past the
//   caches, so the ticket needs no fence (760 keys of 4 kv heads x 256: 10.1 -> 8.3 us).  More splits take
//   a second kernel: draws on one address are served one after the other, 0.15 us each.  A single
//   split writes the output.
//   With a position list (sel[]: the block-sparse decode of src/mm_model.c:1962-2047, whose
//   selected blocks the caller has expanded to positions) list entry i names cache row sel[i];
//   entries that name no row (negative, or beyond n_rows) carry no weight.
#include "common.hpp"
#include "merge.hpp"

namespace cwick {

constexpr int GQA_DEC_THREADS = 256;
constexpr int GQA_DEC_TILE = 16;   // keys per wave and step
constexpr int GQA_DEC_LAST_MERGE = 16;   // splits that the last workgroup of a kv head merges itself

template <int HD>
struct GqaDecTile {
    u32x4 k[HD / 32], v[4][HD / 128];
};

template <int HD, int GROUP>
constexpr int GQA_DEC_QUADS = GROUP <= 4 ? 1 : GROUP == 8 && HD == 128 ? 2 : 0;   // (8 x 256: too many accumulators)

// (Two workgroups per compute unit is what the launcher makes at most; where three fit the registers, they do.
// Eight heads x 128 need 171 registers: held to three, 12 bytes of scratch in the loop, 30000 keys 27.6 us, 26.2 so.)
template <int HD, int GROUP, bool LIST>
__global__ void __launch_bounds__(GQA_DEC_THREADS, HD == 256 || GROUP == 8 ? 2 : 3)
gqa_decode_split_kernel(const uint16_t *__restrict__ K, const uint16_t *__restrict__ V,
                        const uint16_t *__restrict__ Q, int n_keys, int n_kv_heads, int n_splits,
                        float scale_log2e,
                        const int32_t *__restrict__ sel, int64_t n_rows,
                        // (up to here they arrive in registers: what the first loads need is among them)
                        float *__restrict__ part_acc,   // [n_splits][n_heads][HD]
                        float *__restrict__ part_ml,    // [n_splits][n_heads][2]
                        float *__restrict__ out,        // [n_heads][HD], one split only; host memory where there are flags
                        uint32_t *flags, uint32_t epoch,     // a flag per kv head, or null
                        uint32_t *tickets) {            // one per kv head, zero: the last workgroup merges; or null
    constexpr int NW = GQA_DEC_THREADS / 64, NK = HD / 32, NV = HD / 128;
    constexpr int QUADS = GQA_DEC_QUADS<HD, GROUP>, NQ = QUADS > 1 ? QUADS : 1;
    constexpr float SLACK = 64.0f;
    const int g = blockIdx.y, split = blockIdx.x;
    const int n_heads = n_kv_heads * GROUP;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, lg = lane >> 4;
    const uint32_t row_stride = (uint32_t)n_kv_heads * HD;
    const int64_t k_begin = (int64_t)split * (NW * GQA_DEC_TILE);
    const int count = n_keys - (int)k_begin;          // from its first key to the end (negative: none)
    const uint16_t *Kg = K + (LIST ? 0 : k_begin * row_stride) + (size_t)g * HD + lg * 8;
    const uint16_t *Vg = V + (LIST ? 0 : k_begin * row_stride) + (size_t)g * HD + l16 * 8;
    const int32_t *list = LIST ? sel + k_begin : nullptr;

    const int STRIDE = n_splits * (NW * GQA_DEC_TILE);
    int t = wave * GQA_DEC_TILE;
    // List entries, those of four of the wave's tiles in one register: lane 16 j + i has key i of the j-th.
    // A tile takes what it needs (key l16, whose K row this lane reads, and keys 4 lg .. +4 of the V rows)
    // from other lanes when it is requested, and what outlives the request is a bit for each of the four.
    // (Five entries per tile, in registers beside two tiles and waited for one by one: of eight heads x 128
    // and of every group x 256 the loop spilled.  16 blocks of 256 on 8 kv heads x 128, eight query heads
    // each: 10.5 us, 7.2 so; 16 of 128 on 4 x 256, sixteen heads each: 8.4, 7.5.)
    const uint32_t rows_end = (uint32_t)(n_rows < ((int64_t)1 << 31) ? n_rows : (int64_t)1 << 31);
    int32_t names = 0, names_next = 0;
    int j = 4;                                          // tiles of `names` that have been requested
    auto entries = [&](int t) {
        const int i = t + STRIDE * lg + l16;
        return list[i < count ? i : count - 1];
    };
    // Requests a tile and returns which of this lane's keys 4 lg .. +4 carry no weight: those past the end
    // and list entries that name no row, which are read from a row that exists.
    auto load = [&](GqaDecTile<HD> &x, int t) {
        uint32_t k_row, v_row[4], dead = 0;
        if (LIST) {
            if (j == 4) {
                j = 0;
                names = t + STRIDE * lg + l16 < count && (uint32_t)names_next < rows_end ? names_next : -1;
                if (t + 4 * STRIDE < count) names_next = entries(t + 4 * STRIDE);
            }
            const int32_t k = __builtin_amdgcn_ds_bpermute(4 * (16 * j + l16), names);
            k_row = k < 0 ? 0u : (uint32_t)k;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int32_t v = __builtin_amdgcn_ds_bpermute(4 * (16 * j + 4 * lg + r), names);
                v_row[r] = v < 0 ? 0u : (uint32_t)v;
                if (v < 0) dead |= 1u << r;
            }
            j++;
        } else {
            k_row = (uint32_t)(t + l16 < count ? t + l16 : count - 1);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int i = t + 4 * lg + r;
                v_row[r] = (uint32_t)(i < count ? i : count - 1);
                if (i >= count) dead |= 1u << r;
            }
        }
        const uint16_t *kp = Kg + (uint64_t)k_row * row_stride;
#pragma unroll
        for (int i = 0; i < NK; i++) x.k[i] = *(const u32x4 *)(kp + 32 * i);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const uint16_t *vp = Vg + (uint64_t)v_row[r] * row_stride;
#pragma unroll
            for (int h = 0; h < NV; h++) x.v[r][h] = *(const u32x4 *)(vp + 128 * h);
        }
        return dead;
    };
    // The waves of the workgroup meet here at the end; until then a wave's part holds its queries.
    __shared__ __attribute__((aligned(16))) float sh_acc[NW][GROUP][HD];
    // The group's queries come whole, 1 KiB a load, and go through LDS to the lanes (sixteen-byte piece p of head h at
    // place p ^ h, so that the heads of a read come from different banks).  Loads of what each lane needs touch a line
    // for every lane and occupy the memory pipeline as long as the tile behind them, which a workgroup with one tile
    // per wave waits for.  (With the folds below in one statement and no rescale before the first tile, replayed from a
    // graph: 300 keys of 4 x 256 with sixteen heads 7.99 -> 7.04 us, 4096 keys 9.15 -> 8.65; 5000 of 4 x 128 with 32
    // heads 9.12 -> 8.52, 4096 of 8 x 128 with 64 9.13 -> 8.74; 20000 and more keys the same to 1 %.)
    // (Not sixteen heads x 256: as many loads either way, and two registers more than there are.)
    constexpr bool Q_WHOLE = HD * GROUP < 4096;
    constexpr int Q_LOADS = Q_WHOLE ? (GROUP * HD * 2 + 1023) / 1024 : NK;
    constexpr int PIECES = HD / 8;                      // of a head
    u32x4 q_raw[Q_LOADS];
    auto request_q = [&]() {
        if constexpr (!Q_WHOLE) {
#pragma unroll
            for (int j = 0; j < NK; j++) q_raw[j] = *(const u32x4 *)(Q + (size_t)(g * GROUP + l16) * HD + 32 * j + 8 * lg);
            return;
        }
#pragma unroll
        for (int i = 0; i < Q_LOADS; i++) {
            const int piece = 64 * i + lane;
            q_raw[i] = *(const u32x4 *)(Q + (size_t)g * (GROUP * HD) + 8 * (piece < GROUP * PIECES ? piece : 0));
        }
    };
    // this lane's part of the queries: head `col`, dims 32j + 8 lg .. +8
    const int col = QUADS ? l16 % GROUP : l16;
    bf16x8 q[NK];
    auto place_q = [&]() {
        if constexpr (!Q_WHOLE) {
#pragma unroll
            for (int j = 0; j < NK; j++) q[j] = __builtin_bit_cast(bf16x8, q_raw[j]);
            return;
        }
        unsigned char *mine = (unsigned char *)&sh_acc[wave][0][0];
#pragma unroll
        for (int i = 0; i < Q_LOADS; i++) {
            const int piece = 64 * i + lane, h = piece / PIECES;
            if (GROUP * PIECES % 64 == 0 || piece < GROUP * PIECES) *(u32x4 *)(mine + 16 * (piece ^ (h & 15))) = q_raw[i];
        }
        const unsigned char *from = mine + (col < GROUP ? col : 0) * (HD * 2);
#pragma unroll
        for (int j = 0; j < NK; j++) {
            u32x4 w = *(const u32x4 *)(from + 16 * ((4 * j + lg) ^ (col & 15)));
            if (!QUADS && GROUP < 16 && col >= GROUP) w = (u32x4){0u, 0u, 0u, 0u};
            q[j] = __builtin_bit_cast(bf16x8, w);
        }
    };

    // acc[.][8h + i]: dim 128 h + 8 l16 + i; heads 4 lg .. +4, with QUADS heads 4 qd .. +4 over the
    // lane group's keys
    f32x4 acc[NQ][8 * NV];
#pragma unroll
    for (int qd = 0; qd < NQ; qd++)
#pragma unroll
        for (int i = 0; i < 8 * NV; i++) acc[qd][i] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    float m = -INFINITY, l = 0.0f;                      // head `col`; l over this lane's keys

    auto step = [&](const GqaDecTile<HD> &x, uint32_t dead) {
        f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < NK; j++) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x.k[j]), q[j], s, 0, 0, 0);
        float top = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            s[r] = (dead >> r) & 1u ? -INFINITY : s[r] * scale_log2e;
            top = fmaxf(top, s[r]);
        }
        if (__any(top > m + SLACK)) {                   // the first tile, and hardly ever again
            top = fmaxf(m, xor32_max(xor16_max(top)));
            const float corr = top > -INFINITY ? __builtin_amdgcn_exp2f(m - top) : 1.0f;
            const bool some = __any(m > -INFINITY);     // (before that nothing has been added up)
            m = top;
            l *= corr;
            if (some)
#pragma unroll
                for (int qd = 0; qd < NQ; qd++) {
                    f32x4 c;                            // the factors of the accumulators' heads
#pragma unroll
                    for (int r = 0; r < 4; r++) c[r] = __shfl(corr, QUADS ? 4 * qd + r : 4 * lg + r, 64);
#pragma unroll
                    for (int i = 0; i < 8 * NV; i++) acc[qd][i] *= c;
                }
        }
        const float mu = m == -INFINITY ? 0.0f : m;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            s[r] = __builtin_amdgcn_exp2f(s[r] - mu);
            l += s[r];
        }
        auto product = [](float p, float val, f32x4 &d) {
            if (QUADS) d = __builtin_amdgcn_mfma_f32_4x4x1f32(p, val, d, 0, 0, 0);
            else d = __builtin_amdgcn_mfma_f32_16x16x4f32(p, val, d, 0, 0, 0);
        };
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float sr = s[r];          // (a copy: __builtin_bit_cast of a vector's element takes element 0)
            float p[NQ] = {sr};
            if (QUADS == 2) {
                // lanes 4..7 of eight hold heads 4..7: each half's weights to both halves
                const int w = __builtin_bit_cast(int, sr);
                p[0] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(w, w, 0x114, 0xF, 0xA, false));        // row_shr:4
                p[NQ - 1] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(w, w, 0x104, 0xF, 0x5, false));   // row_shl:4
            }
#pragma unroll
            for (int h = 0; h < NV; h++)
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int qd = 0; qd < NQ; qd++) {
                        product(p[qd], bf16lo_to_f32(x.v[r][h][i]), acc[qd][8 * h + 2 * i]);
                        product(p[qd], bf16hi_to_f32(x.v[r][h][i]), acc[qd][8 * h + 2 * i + 1]);
                    }
        }
    };

    if (t < count) {
        GqaDecTile<HD> a, b;
        if (LIST) names_next = entries(t);
        request_q();
        uint32_t dead_a = load(a, t), dead_b = 0;
        place_q();
        for (;;) {
            if (t + STRIDE < count) dead_b = load(b, t + STRIDE);
            step(a, dead_a);
            t += STRIDE;
            if (t >= count) break;
            if (t + STRIDE < count) dead_a = load(a, t + STRIDE);
            step(b, dead_b);
            t += STRIDE;
            if (t >= count) break;
        }
    }
    l = xor32_sum(xor16_sum(l));

    // the waves of the workgroup through LDS
    __shared__ float sh_m[NW][GROUP], sh_l[NW][GROUP];
    if constexpr (QUADS) {
        // the lane groups' sums meet on the way: a swap of two registers leaves one half of the lanes
        // with both parts of the first and the other half with both parts of the second
        // (one statement for four or two swaps: each by itself has two wait states in front of it)
        auto fold32 = [](const float (&x)[4], const float (&y)[4], float *t) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; i++) a[i] = x[i], b[i] = y[i];
            asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %4\n\tv_permlane32_swap_b32 %1, %5\n\tv_permlane32_swap_b32 %2, %6\n\tv_permlane32_swap_b32 %3, %7"
                         : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]));
#pragma unroll
            for (int i = 0; i < 4; i++) t[i] = a[i] + b[i];
        };
        auto fold16 = [](float *t, int half) {          // t[0 .. half) and t[half .. 2 half), half 2 or 4
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; i++) a[i] = t[i % half], b[i] = t[half + i % half];
            if (half == 4)
                asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %4\n\tv_permlane16_swap_b32 %1, %5\n\tv_permlane16_swap_b32 %2, %6\n\tv_permlane16_swap_b32 %3, %7"
                             : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]));
            else
                asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %2\n\tv_permlane16_swap_b32 %1, %3" : "+v"(a[0]), "+v"(a[1]), "+v"(b[0]), "+v"(b[1]));
#pragma unroll
            for (int i = 0; i < half; i++) t[i] = a[i] + b[i];
        };
#pragma unroll
        for (int qd = 0; qd < NQ; qd++)
#pragma unroll
            for (int r = 0; r < (GROUP < 4 ? GROUP : 4); r++) {
                float t[4 * NV];
#pragma unroll
                for (int i = 0; i < 4 * NV; i += 4) {
                    const float x[4] = {acc[qd][i][r], acc[qd][i + 1][r], acc[qd][i + 2][r], acc[qd][i + 3][r]};
                    const float y[4] = {acc[qd][i + 4 * NV][r], acc[qd][i + 4 * NV + 1][r], acc[qd][i + 4 * NV + 2][r], acc[qd][i + 4 * NV + 3][r]};
                    fold32(x, y, t + i);
                }
                fold16(t, 2 * NV);
                // this lane: accumulators 4 NV (lg / 2) + 2 NV (lg % 2) .. + 2 NV
                const int first = 4 * NV * (lg >> 1) + 2 * NV * (lg & 1);
                float *dst = &sh_acc[wave][4 * qd + r][128 * (first >> 3) + 8 * l16 + (first & 7)];
                if constexpr (NV == 2) *(f32x4 *)dst = (f32x4){t[0], t[1], t[2], t[3]};
                else *(f32x2 *)dst = (f32x2){t[0], t[1]};
            }
    } else {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int j = 4 * lg + r;
            if (j < GROUP)
#pragma unroll
                for (int h = 0; h < NV; h++) {
                    const f32x4 *a = &acc[0][8 * h];
                    float *dst = &sh_acc[wave][j][128 * h + 8 * l16];
                    *(f32x4 *)dst = (f32x4){a[0][r], a[1][r], a[2][r], a[3][r]};
                    *(f32x4 *)(dst + 4) = (f32x4){a[4][r], a[5][r], a[6][r], a[7][r]};
                }
        }
    }
    if (lane < GROUP) {
        sh_m[wave][lane] = m;
        sh_l[wave][lane] = l;
    }
    __syncthreads();
    // a thread takes four consecutive dims of one head: the waves' weights once per four values,
    // the values in 16-byte LDS reads, two 8-byte stores
    for (int i4 = threadIdx.x; i4 < GROUP * HD / 4; i4 += GQA_DEC_THREADS) {
        const int j = i4 / (HD / 4), d = (i4 % (HD / 4)) * 4;
        float mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < NW; w++) mx = fmaxf(mx, sh_m[w][j]);
        f32x4 a = {0.0f, 0.0f, 0.0f, 0.0f};
        float ls = 0.0f;
        if (mx > -INFINITY) {
#pragma unroll
            for (int w = 0; w < NW; w++) {
                const float c = __builtin_amdgcn_exp2f(sh_m[w][j] - mx);   // exp2(-inf) = 0 for idle waves
                const f32x4 v = *(const f32x4 *)&sh_acc[w][j][d];
#pragma unroll
                for (int r = 0; r < 4; r++) a[r] = __builtin_fmaf(v[r], c, a[r]);
                ls = __builtin_fmaf(sh_l[w][j], c, ls);
            }
        }
        const int h = g * GROUP + j;
        if (n_splits == 1) {
            a *= ls > 0.0f ? 1.0f / ls : 0.0f;
            if (flags) store_through16(&out[(size_t)h * HD + d], __builtin_bit_cast(u32x4, a));
            else *(f32x4 *)&out[(size_t)h * HD + d] = a;
            continue;
        }
        store_through16(&part_acc[((size_t)split * n_heads + h) * HD + d], __builtin_bit_cast(u32x4, a));
        if (d == 0)
            store_through8(&part_ml[((size_t)split * n_heads + h) * 2], __builtin_bit_cast(u32x2, (f32x2){mx, ls}));
    }
    if (tickets) {
        // The workgroup of the kv head that is through last merges its splits: what they stored is in
        // memory (written through, waited for) when their tickets are drawn, and read past the caches.
        __shared__ uint32_t sh_ticket;
        stores_done();
        __syncthreads();
        if (threadIdx.x == 0) sh_ticket = __hip_atomic_fetch_add(&tickets[g], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (sh_ticket != (uint32_t)n_splits - 1) return;
        if (threadIdx.x == 0) __hip_atomic_store(&tickets[g], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        for (int i4 = threadIdx.x; i4 < GROUP * HD / 4; i4 += GQA_DEC_THREADS) {
            const int h = g * GROUP + i4 / (HD / 4), d = (i4 % (HD / 4)) * 4;
            const float *pa = part_acc + (size_t)h * HD + d, *pm = part_ml + 2 * h;
            f32x2 v[GQA_DEC_LAST_MERGE];
            u32x4 a[GQA_DEC_LAST_MERGE];
#pragma unroll
            for (int s = 0; s < GQA_DEC_LAST_MERGE; s++) {      // (absent splits: the last one again, not counted)
                const int sc = s < n_splits ? s : n_splits - 1;
                v[s] = __builtin_bit_cast(f32x2, __hip_atomic_load((const uint64_t *)(pm + (size_t)sc * n_heads * 2), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM));
                a[s] = load_host16(pa + (size_t)sc * n_heads * HD);
            }
            float mx = -INFINITY, ls = 0.0f;
#pragma unroll
            for (int s = 0; s < GQA_DEC_LAST_MERGE; s++) mx = fmaxf(mx, v[s][0]);
            f32x4 r = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < GQA_DEC_LAST_MERGE; s++) {
                const float c = s < n_splits && v[s][0] > -INFINITY ? __builtin_amdgcn_exp2f(v[s][0] - mx) : 0.0f;
                const f32x4 x = __builtin_bit_cast(f32x4, a[s]);
#pragma unroll
                for (int k = 0; k < 4; k++) r[k] = __builtin_fmaf(x[k], c, r[k]);
                ls = __builtin_fmaf(v[s][1], c, ls);
            }
            r *= ls > 0.0f ? 1.0f / ls : 0.0f;
            if (flags) store_through16(&out[(size_t)h * HD + d], __builtin_bit_cast(u32x4, r));
            else *(f32x4 *)&out[(size_t)h * HD + d] = r;
        }
    }
    if (flags && (tickets || n_splits == 1)) {
        stores_done();
        __syncthreads();
        if (threadIdx.x == 0) host_flag(flags, g, epoch);
    }
}

template <int HD, int GROUP>
static int run_gqa_decode(const uint16_t *k, const uint16_t *v, int64_t n_keys, int n_kv_heads,
                          const int32_t *sel, int64_t n_rows, const uint16_t *q, float scale, float *out,
                          hipStream_t s, HostFlags *done) {
    const int n_heads = n_kv_heads * GROUP;
    constexpr int step = (GQA_DEC_THREADS / 64) * GQA_DEC_TILE;     // keys a workgroup takes at a time
    // One workgroup per compute unit with an equal share of steps: its four waves and the tiles they
    // have requested ahead saturate the unit's path to memory, and more workgroups only add partials
    // (16384 keys on 4 kv heads x 256: 17.7 us with 256 workgroups, 19.2 with 512; 100003 on
    // 8 x 128: 79 and 85).  Where two workgroups per unit make it a single step each, that is the
    // shorter (4096 keys on 8 x 128: 8.9 against 9.5), and up to three steps in one workgroup are
    // shorter than a second launch (100 keys: 6.8 against 8.2).
    const int64_t steps = (n_keys + step - 1) / step;
    int64_t per_steps = 1;
    if (steps <= 3) per_steps = steps;
    else if (steps * n_kv_heads > 2 * num_cus()) {
        const int64_t want = num_cus() > n_kv_heads ? num_cus() / n_kv_heads : 1;
        per_steps = (steps + want - 1) / want;
    }
    const int n_splits = (int)((steps + per_steps - 1) / per_steps);
    float *part_acc = nullptr, *part_ml = nullptr;
    if (n_splits > 1) {
        // (asked for: as many splits as any call of up to this many keys has)
        const int64_t single = 2 * num_cus() / n_kv_heads, most = steps < single ? steps : single;
        const size_t per_split = (size_t)n_heads * (HD + 2) * sizeof(float);
        char *ws = (char *)workspace(s, (size_t)(most > n_splits ? most : n_splits) * per_split);
        if (!ws) return 0;                  // workspace() has recorded why
        part_acc = (float *)ws, part_ml = part_acc + (size_t)n_splits * n_heads * HD;
    }
    uint32_t *flags = done ? done->flags : nullptr;
    const uint32_t epoch = done ? done->epoch : 0u;
    uint32_t *tickets = nullptr;            // (a stream that has none yet and is being captured merges in a second launch)
    if (n_splits > 1 && n_splits <= GQA_DEC_LAST_MERGE) tickets = ticket_counters_if_free(s);
    const bool one_launch = n_splits == 1 || tickets;
    if (done) done->count = one_launch ? n_kv_heads : n_heads;
    {
        ProfKernel pk(CWICK_HIP_PROF_GQA_DECODE, s);
        pk.launch(sel ? gqa_decode_split_kernel<HD, GROUP, true> : gqa_decode_split_kernel<HD, GROUP, false>,
                  dim3(n_splits, n_kv_heads), dim3(GQA_DEC_THREADS), 0, k, v, q, (int)n_keys, n_kv_heads, n_splits,
                  scale * 1.44269504088896340736f, sel, n_rows, part_acc, part_ml, out, flags, epoch, tickets);
    }
    CWICK_HIP_CALL(hipGetLastError());
    if (one_launch) return 1;
    {
        ProfKernel pk(CWICK_HIP_PROF_GQA_DECODE_MERGE, s);
        pk.launch(splitk_merge_wide_kernel<HD>, dim3(n_heads, 1), dim3(64 * (n_splits < 16 ? n_splits : 16)), 0,
                  part_acc, part_ml, n_splits, n_heads, out, flags, epoch);
    }
    CWICK_HIP_CALL(hipGetLastError());
    return 1;
}

int launch_gqa_decode(const uint16_t *k, const uint16_t *v, int64_t n_keys, int n_kv_heads,
                      int head_dim, const uint16_t *q, int n_heads, float scale, float *out,
                      hipStream_t s, const int32_t *sel, int64_t n_rows, HostFlags *done) {
    CWICK_REQUIRE(k && v && q && out, "gqa_decode: null pointer");
    CWICK_REQUIRE(n_keys >= 1 && n_keys <= ((int64_t)1 << 30), "gqa_decode: n_keys %lld",
                  (long long)n_keys);
    CWICK_REQUIRE(n_kv_heads >= 1 && n_kv_heads <= 64 && n_heads >= n_kv_heads &&
                      n_heads % n_kv_heads == 0,
                  "gqa_decode: n_heads %d is not a multiple of n_kv_heads %d", n_heads, n_kv_heads);
    CWICK_REQUIRE(((uintptr_t)k | (uintptr_t)v | (uintptr_t)q) % 16 == 0,
                  "gqa_decode: K, V and q must be 16-byte aligned");
    const int group = n_heads / n_kv_heads;
#define CASE(HD, G)                                      \
    if (head_dim == HD && group == G)                    \
        return run_gqa_decode<HD, G>(k, v, n_keys, n_kv_heads, sel, n_rows, q, scale, out, s, done)
    CASE(256, 1); CASE(256, 2); CASE(256, 4); CASE(256, 8); CASE(256, 16);
    CASE(128, 1); CASE(128, 2); CASE(128, 4); CASE(128, 8); CASE(128, 16);
#undef CASE
    set_error("gqa_decode: head_dim %d with group %d is not supported (head_dim 128/256, group 1/2/4/8/16)",
              head_dim, group);
    return 0;
}

}  // namespace cwick
