// gqa_prefill.hip -- causal GQA prefill on the bf16 matrix cores (the prefill
// branch of the reference's mixer_attn, src/q35_model.c:1713-1746: per head and
// per 128-query tile S = scale*Q*K^T over the rectangle, -1e30 tail, softmax,
// O = S*V).  Here: one pass, online softmax, the triangle only.
//
// MFMA-bound, and on this machine that means LDS-aware: a 32x32x16 MFMA takes
// 32 cycles and its A operand is 1 KiB, so four SIMDs that each fetch their own
// A fragments need the whole 128 B/clk of LDS.  Every wave therefore owns 64
// query rows (two 32-row column blocks) and uses each K / V^T fragment twice.
//
//   workgroup = 4 waves = 256 query rows that share one kv head: the GROUP
//   query heads of the kv head times P = 256/GROUP consecutive positions
//   (heads-as-M: K and V tiles are read once for all heads of the group).
//   Key tiles of TK = 32.  K and V go global -> LDS by global_load_lds_dwordx4
//   (no staging registers), one workgroup barrier per tile.
//   scores:  S^T[key][row] = K[key][dim] . Q^T[dim][row], v_mfma_f32_32x32x16_bf16,
//            K fragments from LDS, Q fragments of the first column block resident in
//            registers, those of the second re-read from a per-lane LDS park.
//            One query row per lane column: softmax statistics are per-lane.
//            The score accumulators are pinned to VGPRs (inline assembly): through the
//            builtin every MFMA result is placed in AGPRs, which the outputs fill.
//   values:  O^T[dim][row] += V^T[dim][key] . P^T[key][row].  P^T is the score
//            accumulator itself (rounded to bf16) -- its register layout is the
//            B-operand layout once the contraction slots are numbered to match;
//            V^T fragments come out of the V tile through the LDS transpose read
//            (ds_read_b64_tr_b16).  The 256 output registers live in AGPRs.
//   schedule: one wave per SIMD, so the loop is software-pipelined by hand, three
//            tiles deep: step t interleaves, MFMA by MFMA, the scores of tile t+2, the
//            softmax of tile t+1 (VALU, in the shadow of the matrix instructions) and
//            the value products of tile t.  The barrier that opens step t+1 sits near
//            the end of step t and the first fragments of step t+1 are fetched behind
//            it, so the matrix pipe does not drain between steps.  K is copied three
//            tiles ahead into two buffers, V two tiles ahead into three: a tile costs
//            about 500 cycles of the CU's copy path, so the copies are spread over the
//            whole step and only K has to land within it.
//   The softmax reference of a row is the maximum of its first tile and stays
//   there while later scores exceed it by less than 64 (log2 units): weights up
//   to 2^64 lose nothing in bf16 or fp32.  A wave that meets a larger score
//   leaves the fast loop for a slow one that moves the reference and rescales
//   the accumulators (in place, in AGPRs) every tile.
//   Position blocks that see at most 1024 keys run the PRECISE variant (the
//   rounding residual of the weights goes through the matrix core too) in the
//   simpler two-stage schedule: scores of tile t+1, then its softmax next to
//   the value products of tile t.
//
//   Problems that do not fill the chip take gqa_prefill_team_kernel: four waves on 64 rows, each on key tiles of
//   its own.
#include "common.hpp"
#include "gqa_plan.hpp"

#include <mutex>
#include <type_traits>

namespace cwick {

constexpr int PF_HD = 256;
constexpr int PF_WAVES = 4;                 // waves per workgroup
constexpr int PF_PAIR = 1024 + 32;          // bytes between pairs of rows in LDS
constexpr int PF_TILE = 16 * PF_PAIR;       // one K or V tile, or the 32 query rows of a column block, in LDS
constexpr int PF_PRE = 4;                   // k-steps of fragment prefetch in the score loop

typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) void pf_lds_void;

struct PfSmem {
    unsigned char k[2][PF_TILE];
    unsigned char v[3][PF_TILE];                // the pipelined body keeps three V tiles, the other two
    // the query rows of column block B: the register file holds 256 accumulators + 64 Q registers +
    // the working set, not 128 Q registers
    unsigned char q[PF_WAVES][PF_TILE];
};

// A tile in LDS is sixteen pairs of rows, m and m + 16, each row whole (512 bytes), 32 bytes between the
// pairs; in rows with bit 3 set the two 16-byte columns of every 32 bytes are swapped.  A copy
// instruction then fetches two whole rows (8 cache lines; one that fetches a piece of 32 rows occupies
// the memory pipe for 32 to 64 cycles, this one for 16), sixteen neighbouring rows of a fragment read
// fall into different banks, and so do the four rows of a transpose read; and every fragment is at a
// constant distance from its lane's first (a swizzle that XORs more bits cost 72 instructions a tile in a
// loop that is bound by the wave's issue: 486 us instead of 452 for 8192 positions).
__device__ __forceinline__ uint32_t pf_row(uint32_t row) { return (row & 15) * PF_PAIR + (row >> 4) * 512; }
__device__ __forceinline__ uint32_t pf_swap(uint32_t row) { return (row >> 3) & 1; }

// workgroup barrier that orders LDS traffic only (the copies of later tiles stay in flight)
#define PF_LDS_BARRIER() asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory")

// Of the sum of a row's weights.  A score that overflows when it is scaled leaves a reference of infinity and weights of
// zero: its row is NaN, as with a score that overflows by itself and where slices or waves meet (infinity minus infinity).
__device__ __forceinline__ float pf_reciprocal(float l, float m_ref) {
    return m_ref == INFINITY ? __builtin_nanf("") : l > 0.0f ? 1.0f / l : 0.0f;
}

// PRECISE: the bf16 rounding residual of the weights goes through the matrix core as well
// (position blocks that see at most 1024 keys; see the launcher).  The body of one workgroup.
// K and V start at the first key of the item's slice and pos0 counts from there (a whole item: the
// first row, the chunk's own pos0); wg_keys keys of it are the item's.  SPLIT: a slice of a block leaves
// its unnormalised accumulators in register order at slice->part, the rows' reference and weight sum
// at slice->part_ml (in LDS until the end: held in registers they cost the loop its last free ones).
struct PfSlice {
    float *part, *part_ml;                      // part is null for a block that is one slice
};
template <int GROUP, bool PRECISE, bool SPLIT>
__device__ __forceinline__ void
gqa_prefill_body(unsigned char *smem_raw, const uint16_t *__restrict__ K, const uint16_t *__restrict__ V,
                 const uint16_t *__restrict__ Q, int64_t pos0, int64_t n, int64_t wg_keys, int n_kv_heads,
                 float scale_log2e, float *__restrict__ out, int64_t pblk, int kvh,
                 const PfSlice *slice = nullptr) {
    constexpr int P = 64 * PF_WAVES / GROUP;    // positions per workgroup
    constexpr int NI = 16 / PF_WAVES;       // copies of a tile that each wave issues
    PfSmem &sm = *reinterpret_cast<PfSmem *>(smem_raw);

    // The thread's number is opaque to the compiler here, and the copy's key below: what it knows of
    // their ranges and of the loop over items around this body it turns into per-lane constants that
    // live, and spill, across the pipelined loop.
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31;
    const int g = lane >> 5;                // 0/1

    const int64_t t0 = pblk * P;
    const int n_heads = n_kv_heads * GROUP;
    const int64_t q_stride = (int64_t)n_heads * PF_HD;
    const int n_tiles = (int)((wg_keys + PF_TK - 1) / PF_TK);
    const int64_t first_masked_key = pos0 + t0;   // tiles ending at or below this need no mask
    constexpr bool precise = PRECISE;

    // ---- global -> LDS copies.  Copy i of wave w takes rows m and m + 16 of a tile, m = NI w + i: lane l
    // row m + 16 (l>>5), and the column that belongs into column l&31 of that row in LDS.  What lies
    // behind the item's last key (masked anyway) repeats the last 16 bytes of it.
    const uint32_t row_bytes = (uint32_t)n_kv_heads * (PF_HD * 2);
    uint32_t cp_off = (uint32_t)(NI * wave + 16 * g) * row_bytes + (uint32_t)(l32 ^ (NI * wave >> 3)) * 16;
    asm volatile("" : "+v"(cp_off));
    const unsigned char *Kg = (const unsigned char *)(K + (size_t)kvh * PF_HD);
    const unsigned char *Vg = (const unsigned char *)(V + (size_t)kvh * PF_HD);
    const uint32_t lds_k = (uint32_t)(uintptr_t)(pf_lds_void *)&sm.k[0][0];
    const uint32_t lds_v = (uint32_t)(uintptr_t)(pf_lds_void *)&sm.v[0][0];
    const uint32_t lds_q = (uint32_t)(uintptr_t)(pf_lds_void *)&sm.q[wave][0];
    struct CopySrc {
        const unsigned char *base;                              // first row of the tile
        uint32_t last;                                          // byte offset of the last 16 bytes there are
    };
    auto copy_src = [&](const unsigned char *base, int tile) -> CopySrc {
        tile = __builtin_amdgcn_readfirstlane(tile < n_tiles ? tile : n_tiles - 1);     // past the last tile: into a dead buffer
        const uint32_t left = (uint32_t)wg_keys - 1 - (uint32_t)tile * PF_TK;
        const uint64_t first = (uint64_t)base + (uint64_t)((uint32_t)tile * PF_TK) * row_bytes;
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)first), hi = __builtin_amdgcn_readfirstlane((uint32_t)(first >> 32));
        return {(const unsigned char *)((uint64_t)hi << 32 | lo), (left < PF_TK ? left : PF_TK - 1) * row_bytes + (PF_HD * 2 - 16)};
    };
    auto copy_one = [&](const CopySrc &src, uint32_t lds_tile, int i) {
        const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds_tile + (uint32_t)((NI * wave + i) * PF_PAIR));
        uint32_t off = cp_off + (uint32_t)i * row_bytes;
        off = off < src.last ? off : src.last;
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(src.base), "s"(m0) : "memory");
    };
    auto issue = [&](const unsigned char *base, uint32_t lds_tile, int tile) {
        const CopySrc src = copy_src(base, tile);
#pragma unroll
        for (int i = 0; i < NI; i++) copy_one(src, lds_tile, i);
    };

    // The first tiles are requested with the query rows: one trip to memory for all of them
    // instead of one for Q, one for tile 0 and one for tile 1 (K has two buffers, V at least two).
    issue(Kg, lds_k, 0);
    issue(Vg, lds_v, 0);
    if (n_tiles > 1) {
        issue(Kg, lds_k + PF_TILE, 1);
        if (!precise) issue(Vg, lds_v + PF_TILE, 1);
    }

    // The wave's 64 query rows, copied along the rows as K and V are: 32 pieces of 16 B fetched down the
    // rows took the memory pipe as long as seven tiles.  Column block A goes through the LDS place of
    // block B on its way into fragments, block B through registers.
    bf16x8 qf[16];                          // B operand: lane (row, g) holds dims 16ks+8g .. +8
    {
        auto q_src = [&](int c, int m) -> const unsigned char * {
            const int r = wave * 64 + 32 * c + m + 16 * g;
            const int64_t left = n - 1 - t0;
            const uint32_t t = (uint32_t)(r % P) < left ? (uint32_t)(r % P) : (uint32_t)left;
            return (const unsigned char *)(Q + t0 * q_stride + (size_t)kvh * GROUP * PF_HD) +
                   (uint64_t)t * ((uint32_t)n_heads * (PF_HD * 2)) + (r / P) * (PF_HD * 2) + ((uint32_t)l32 ^ pf_swap(m)) * 16;
        };
#pragma unroll
        for (int m = 0; m < 16; m++) {
            const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds_q + m * PF_PAIR);
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(q_src(0, m)), "s"(m0) : "memory");
        }
        u32x4 qb[16];
#pragma unroll
        for (int m = 0; m < 16; m++) qb[m] = *(const u32x4 *)q_src(1, m);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const unsigned char *a = &sm.q[wave][pf_row(l32) + ((g ^ pf_swap(l32)) << 4)];
#pragma unroll
        for (int ks = 0; ks < 16; ks++) qf[ks] = __builtin_bit_cast(bf16x8, *(const u32x4 *)(a + 32 * ks));
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int m = 0; m < 16; m++) *(u32x4 *)&sm.q[wave][m * PF_PAIR + lane * 16] = qb[m];
    }

    // K fragment of k-step ks: row l32, column 2ks + g; so for the query rows of block B
    const unsigned char *kfrag = &sm.k[0][pf_row(l32) + ((g ^ pf_swap(l32)) << 4)];
    const unsigned char *qfrag = &sm.q[wave][pf_row(l32) + ((g ^ pf_swap(l32)) << 4)];
    // transpose read (ds_read_b64_tr_b16): within a 16-lane group, lane i addresses key (i/4),
    // dims 4*(i%4)..+4 of a 4-key x 16-dim patch and receives dim i for the 4 keys.
    // For output block db: dims 32db + 16(grp&1) + 4(gi&3): column c = 4db + 2(grp&1) + ((gi&3)>>1)
    const int grp = lane >> 4, gi = lane & 15;
    const int v_key0 = 4 * (grp >> 1) + (gi >> 2);                // + 16 ks2 (+8 for the second half)
    const int v_col = 2 * (grp & 1) + ((gi & 3) >> 1);
    const unsigned char *vfrag[2] = {&sm.v[0][pf_row(v_key0) + (v_col << 4) + (gi & 1) * 8],
                                     &sm.v[0][pf_row(v_key0 + 8) + ((v_col ^ 1) << 4) + (gi & 1) * 8]};
    // step st of a value product: 32 dims (st & 7) of the 16 keys st >> 3, in two halves
    auto vread = [&](int off, int st, int half) -> s16x4 {
        return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(vfrag[half] + off + (st & 7) * 64 + (st >> 3) * 512));
    };

    f32x16 oacc[2][8];
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
        for (int db = 0; db < 8; db++)
#pragma unroll
            for (int i = 0; i < 16; i++) oacc[c][db][i] = 0.0f;
    float m_ref[2] = {-INFINITY, -INFINITY}, l_part[2] = {0.0f, 0.0f};

    // scores of one tile for both column blocks
    // One wave per SIMD: nothing hides an LDS round trip, so the fragments are fetched PF_PRE
    // k-steps ahead of the MFMAs that use them.
    // Score MFMA with its accumulator pinned to VGPRs: through the builtin the allocator places
    // every MFMA result in AGPRs, which the 256 output accumulators fill, and moves registers
    // back and forth every tile.  Opaque to the compiler's hazard tracking: score_done() goes
    // between the last MFMA and the first VALU read of the result, and carries the result (without,
    // nothing keeps the first instruction that reads it behind the wait).
    auto score_mfma = [&](f32x16 &acc, bf16x8 a, bf16x8 b, bool first) {
        if (first) asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(acc) : "v"(a), "v"(b));
        else asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b));
    };
    auto score_done = [&](f32x16 (&s)[2]) { asm volatile("s_nop 15\n\ts_nop 15" : "+v"(s[0]), "+v"(s[1])::"memory"); };
    // ck / cv >= 0: the copies of K(ck) and V(cv) are issued between the MFMAs (an LDS-DMA
    // instruction occupies the issue slot for about as long as two MFMAs run).  Tile u of K or V
    // lives in buffer u & 1.
    auto scores = [&](int tile, f32x16 (&s)[2], int ck, int cv) {
        const unsigned char *kb = kfrag + (tile & 1) * PF_TILE;
        u32x4 ka[PF_PRE], qa[PF_PRE];
#pragma unroll
        for (int ks = 0; ks < PF_PRE; ks++) {
            ka[ks] = *(const u32x4 *)(kb + 32 * ks);
            qa[ks] = *(const u32x4 *)(qfrag + 32 * ks);
        }
        const bool do_k = ck >= 0 && ck < n_tiles, do_v = cv >= 0 && cv < n_tiles;
        const CopySrc src_k = copy_src(Kg, do_k ? ck : 0), src_v = copy_src(Vg, do_v ? cv : 0);
        const uint32_t dst_k = lds_k + (uint32_t)((ck & 1) * PF_TILE);
        const uint32_t dst_v = lds_v + (uint32_t)((cv & 1) * PF_TILE);
#pragma unroll
        for (int ks = 0; ks < 16; ks++) {
            const bf16x8 kf = __builtin_bit_cast(bf16x8, ka[ks % PF_PRE]);
            const bf16x8 q1 = __builtin_bit_cast(bf16x8, qa[ks % PF_PRE]);
            if (ks + PF_PRE < 16) {
                ka[ks % PF_PRE] = *(const u32x4 *)(kb + 32 * (ks + PF_PRE));
                qa[ks % PF_PRE] = *(const u32x4 *)(qfrag + 32 * (ks + PF_PRE));
            }
            score_mfma(s[0], kf, qf[ks], ks == 0);
            score_mfma(s[1], kf, q1, ks == 0);
#pragma unroll
            for (int i = (ks & 7) * NI / 8; i < ((ks & 7) + 1) * NI / 8; i++) {
                if (ks < 8) { if (do_k) copy_one(src_k, dst_k, i); }
                else if (do_v) copy_one(src_v, dst_v, i);
            }
        }
        score_done(s);
    };
    // the same from global memory (the slow loop of the pipelined body: its K tile has already
    // been overwritten in LDS)
    auto scores_global = [&](int tile, f32x16 (&s)[2]) {
        int64_t row = (int64_t)tile * PF_TK + l32;
        if (row > wg_keys - 1) row = wg_keys - 1;                   // masked anyway
        const uint16_t *kr = (const uint16_t *)(Kg + row * row_bytes) + 8 * g;
#pragma unroll
        for (int ks = 0; ks < 16; ks++) {
            const bf16x8 kf = __builtin_bit_cast(bf16x8, *(const u32x4 *)(kr + 16 * ks));
            const bf16x8 q1 = __builtin_bit_cast(bf16x8, *(const u32x4 *)(qfrag + 32 * ks));
            score_mfma(s[0], kf, qf[ks], ks == 0);
            score_mfma(s[1], kf, q1, ks == 0);
        }
        score_done(s);
    };
    // softmax bookkeeping of one tile and column block, in two parts.
    // register i holds key (i/4)*8 + 4g + i%4 of the tile for this lane's row.
    // sm_prep: mask the raw scores, return this lane's maximum in log2 units.
    auto sm_prep = [&](int tile, int c, f32x16 &s) -> float {
        const int64_t key0 = (int64_t)tile * PF_TK;
        float tmax = -INFINITY;
        if (key0 + PF_TK - 1 > first_masked_key) {          // workgroup-uniform: a tile on the diagonal
            // position (i/4)*8 + i%4 + 4g of the tile is visible up to lim (rows behind the chunk's last
            // position take part as that one)
            const int left = (int)(n - 1 - t0 < P ? n - 1 - t0 : P), tr = (wave * 64 + 32 * c + l32) % P;
            const int lim = (int)(first_masked_key - key0) + (tr < left ? tr : left) - 4 * g;
#pragma unroll
            for (int i = 0; i < 16; i++)
                if ((i >> 2) * 8 + (i & 3) > lim) s[i] = -INFINITY;
        }
#pragma unroll
        for (int i = 0; i < 16; i++) tmax = fmaxf(tmax, s[i]);
        return tmax * scale_log2e;                           // the scale is positive: max commutes
    };
    // sm_finish: raw scores -> bf16 weights (and their rounding residual) against m_ref.
    auto sm_finish = [&](int c, f32x16 &s, u32x4 (&pw)[2], u32x4 (&pl)[2]) {
        const float m_use = m_ref[c] == -INFINITY ? 0.0f : m_ref[c];
        float psum = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            s[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], scale_log2e, -m_use));   // masked: 0
            if (precise) psum += s[i];
        }
        // contraction slot (g, jj) of step ks2 <-> tile key 16*ks2 + (jj/4)*8 + 4g + jj%4,
        // i.e. score register 8*ks2 + jj: P^T needs no data movement.
        // With single-term weights the row sum is the sum of the ROUNDED weights: the output is
        // then a convex combination of value rows whatever the rounding did (a row dominated by
        // one key is exact), and the error is 2^-9 of the spread of the values, not of their size.
#pragma unroll
        for (int ks2 = 0; ks2 < 2; ks2++)
#pragma unroll
            for (int h = 0; h < 4; h++) {
                pw[ks2][h] = pack_bf16_rne(s[8 * ks2 + 2 * h], s[8 * ks2 + 2 * h + 1]);
                if (precise)
                    pl[ks2][h] = pack_bf16_rne(s[8 * ks2 + 2 * h] - bf16lo_to_f32(pw[ks2][h]),
                                               s[8 * ks2 + 2 * h + 1] - bf16hi_to_f32(pw[ks2][h]));
                else
                    psum = pair_sum_bf16(pw[ks2][h], psum);
            }
        l_part[c] += psum;
    };
    // The running reference m_ref is the row maximum of tile 0 and stays there while later tiles
    // exceed it by less than 2^SLACK: weights up to 2^SLACK are as exact in bf16 and fp32 as
    // weights up to 1.  The slow loop moves it (and rescales) when a tile beats it by 2^8.
    constexpr float SLACK = 64.0f;
    auto sm_move_ref = [&](int c, float tmax) -> float {
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
        float corr = 1.0f;
        if (tmax > m_ref[c] + 8.0f) {
            corr = __builtin_amdgcn_exp2f(m_ref[c] - tmax);              // first tile: exp2(-inf) = 0
            m_ref[c] = tmax;
            l_part[c] *= corr;
        }
        return corr;
    };
    // value MFMAs of one tile for both column blocks
    auto values = [&](int tile, const u32x4 (&pw)[2][2], const u32x4 (&pl)[2][2]) {
        const int vb = (PRECISE ? (tile & 1) : (tile % 3)) * PF_TILE;
        // step st = 8 ks2 + db; its two transpose reads are issued PF_PRE steps ahead
        s16x4 lo[PF_PRE], hi[PF_PRE];
        auto fetch = [&](int st, int slot) {
            lo[slot] = vread(vb, st, 0);
            hi[slot] = vread(vb, st, 1);
        };
#pragma unroll
        for (int st = 0; st < PF_PRE; st++) fetch(st, st);
#pragma unroll
        for (int st = 0; st < 16; st++) {
            const int ks2 = st >> 3, db = st & 7;
            typedef __attribute__((ext_vector_type(8))) short s16x8;
            const bf16x8 va = __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(lo[st % PF_PRE], hi[st % PF_PRE], 0, 1, 2, 3, 4, 5, 6, 7));
            if (st + PF_PRE < 16) fetch(st + PF_PRE, st % PF_PRE);
#pragma unroll
            for (int c = 0; c < 2; c++) {
                oacc[c][db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, __builtin_bit_cast(bf16x8, pw[c][ks2]), oacc[c][db], 0, 0, 0);
                if (precise)
                    oacc[c][db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, __builtin_bit_cast(bf16x8, pl[c][ks2]), oacc[c][db], 0, 0, 0);
            }
        }
    };
    // The accumulators live in AGPRs.  Written as ordinary arithmetic a rescale makes the
    // compiler move them to VGPRs for the whole loop (and spill), and so does a rescale under a
    // condition; so the fast loop has none, and the slow loop scales every tile, in place.
    auto rescale = [&](const float (&corr)[2]) {
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int db = 0; db < 8; db++)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    float tmp;
                    asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\ts_nop 0\n\t"
                                 "v_accvgpr_write_b32 %0, %1"
                                 : "+a"(oacc[c][db][i]), "=&v"(tmp)
                                 : "v"(corr[c]));
                }
    };
    // top of step t: the tiles step t reads have landed (this wave's part, then everyone's), and
    // all reads of step t-1 are over, so the copies of step t may overwrite its buffers
    auto step_top = [&]() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        PF_LDS_BARRIER();
    };

    if constexpr (PRECISE) {
        // ---- prologue: K(0), V(0), K(1) are on their way; scores and softmax of tile 0 (sets the reference) ----
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        PF_LDS_BARRIER();

        u32x4 pw[2][2], pl[2][2];
        {
            f32x16 s[2];
            scores(0, s, -1, -1);
#pragma unroll
            for (int c = 0; c < 2; c++) {
                (void)sm_move_ref(c, sm_prep(0, c, s[c]));                  // nothing accumulated yet
                sm_finish(c, s[c], pw[c], pl[c]);
            }
        }

        // ---- fast loop: scores(t+1); then softmax(t+1) beside values(t); no rescale.  The softmax
        // is speculative: whether a row outgrew the reference is looked at after the MFMAs.
        int t = 0;
        bool slow = false;
        for (; t + 1 < n_tiles; t++) {
            step_top();
            f32x16 s[2];
            scores(t + 1, s, t + 2, t + 1);
            u32x4 pwn[2][2], pln[2][2];
            const float l_save[2] = {l_part[0], l_part[1]};
            const float x0 = sm_prep(t + 1, 0, s[0]), x1 = sm_prep(t + 1, 1, s[1]);
            sm_finish(0, s[0], pwn[0], pln[0]);
            sm_finish(1, s[1], pwn[1], pln[1]);
            values(t, pw, pl);
            if (__any(x0 > m_ref[0] + SLACK || x1 > m_ref[1] + SLACK)) {   // a row outgrew the reference
                l_part[0] = l_save[0];
                l_part[1] = l_save[1];
                slow = true;
                break;
            }
#pragma unroll
            for (int c = 0; c < 2; c++)
#pragma unroll
                for (int k2 = 0; k2 < 2; k2++) {
                    pw[c][k2] = pwn[c][k2];
                    pl[c][k2] = pln[c][k2];
                }
        }
        // ---- slow loop (rare): the reference follows the maximum, accumulators rescaled every tile.
        // It resumes step t after its top, copies and values(t); the scores are recomputed.
        if (slow) {
            bool resumed = true;
            for (; t + 1 < n_tiles; t++) {
                if (!resumed) step_top();
                f32x16 s[2];
                scores(t + 1, s, resumed ? -1 : t + 2, resumed ? -1 : t + 1);
                u32x4 pwn[2][2], pln[2][2];
                float corr[2];
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    corr[c] = sm_move_ref(c, sm_prep(t + 1, c, s[c]));
                    sm_finish(c, s[c], pwn[c], pln[c]);
                }
                if (!resumed) values(t, pw, pl);
                resumed = false;
                rescale(corr);
#pragma unroll
                for (int c = 0; c < 2; c++)
#pragma unroll
                    for (int k2 = 0; k2 < 2; k2++) {
                        pw[c][k2] = pwn[c][k2];
                        pl[c][k2] = pln[c][k2];
                    }
            }
        }
        // ---- last tile's values ----
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        PF_LDS_BARRIER();
        values(n_tiles - 1, pw, pl);

    } else {
        // ---- pipelined body: step t computes the scores of tile t+2, the softmax of tile t+1 and the
        // value products of tile t, interleaved MFMA by MFMA so that the softmax (VALU), the fragment
        // reads (LDS) and the copies issue in the shadow of the matrix instructions.  The loop is
        // rotated: the barrier that opens step t+1 sits in slot 14 of step t (by then every
        // fragment read of step t has returned and the copies issued in slots 0..7 have landed), and
        // slots 14 and 15 already fetch the first fragments of step t+1, so the matrix pipe does not
        // drain between steps.  Only tiles below the diagonal take this form; the (at most three)
        // tiles on it and the tail run in sequence.
        constexpr float BIG = 18446744073709551616.0f;                  // 2^SLACK
        u32x4 ka[2], qa[2];                                             // fragments of the next two slots
        s16x4 lo[2], hi[2];
        // V(t) lives in buffer t mod 3, carried along as t3 (no division in the loop)
        auto next3 = [](int x) -> int { return x == 2 ? 0 : x + 1; };
        int t3 = 0;
        auto fetch = [&](int t, int t3, int i, int slot) {              // fragments of slot i of step t
            ka[slot] = *(const u32x4 *)(kfrag + (t & 1) * PF_TILE + 32 * i);        // K(t+2)
            qa[slot] = *(const u32x4 *)(qfrag + 32 * i);
            lo[slot] = vread(t3 * PF_TILE, i, 0);                                   // V(t)
            hi[slot] = vread(t3 * PF_TILE, i, 1);
        };
        // the running sums as opaque instructions: left to the compiler, the thirty-two additions
        // of a step sink to its end, a dependent chain behind the last MFMA
        // (one dot-product instruction per packed pair: acc += lo * 1 + hi * 1)
        const uint32_t ones_bf16 = 0x3F803F80u;
        auto psum_pair = [&](float &acc, uint32_t w) { asm volatile("v_dot2c_f32_bf16 %0, %1, %2" : "+v"(acc) : "s"(ones_bf16), "v"(w)); };
        auto pstep = [&](int t, int t3, f32x16 (&sc)[2], f32x16 (&sn)[2], const u32x4 (&pc)[2][2],
                         u32x4 (&pn)[2][2], float (&ps)[2]) {
            const int t3n = next3(t3);
            CopySrc src_k = {nullptr, 0}, src_v = {nullptr, 0};
            uint32_t dst_k = 0, dst_v = 0;
            const float mu0 = m_ref[0], mu1 = m_ref[1];
            float p0 = 0.0f, p1 = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                typedef __attribute__((ext_vector_type(8))) short s16x8;
                const int ks2 = i >> 3, db = i & 7;
                const bf16x8 kf = __builtin_bit_cast(bf16x8, ka[i & 1]);
                const bf16x8 q1 = __builtin_bit_cast(bf16x8, qa[i & 1]);
                const bf16x8 va = __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(lo[i & 1], hi[i & 1], 0, 1, 2, 3, 4, 5, 6, 7));
                score_mfma(sn[0], kf, qf[i], i == 0);
                sc[0][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[0][i], scale_log2e, -mu0));
                if (i == 0) {
                    // where this step's copies come from and go to, worked out behind the
                    // first MFMA
                    src_k = copy_src(Kg, t + 3);
                    src_v = copy_src(Vg, t + 2);
                    dst_k = lds_k + (uint32_t)(((t + 1) & 1) * PF_TILE);
                    dst_v = lds_v + (uint32_t)(next3(t3n) * PF_TILE);
                }
                __builtin_amdgcn_sched_barrier(0);
                oacc[0][db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, __builtin_bit_cast(bf16x8, pc[0][ks2]), oacc[0][db], 0, 0, 0);
                sc[1][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[1][i], scale_log2e, -mu1));
                __builtin_amdgcn_sched_barrier(0);
                score_mfma(sn[1], kf, q1, i == 0);
                if (i == 14) {                                       // the top of step t+1
                    // all but this step's V copies of slots 8 to 13: K(t+3) and V(t+1) have landed
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NI * 3 / 4) : "memory");
                    PF_LDS_BARRIER();
                }
                if (i < 14) fetch(t, t3, i + 2, i & 1);
                else fetch(t + 1, t3n, i - 14, i & 1);
                __builtin_amdgcn_sched_barrier(0);
                oacc[1][db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, __builtin_bit_cast(bf16x8, pc[1][ks2]), oacc[1][db], 0, 0, 0);
                if (i & 1) {                                         // weights, and the sum of the rounded weights
                    const uint32_t w0 = pack_bf16_rne(sc[0][i - 1], sc[0][i]);
                    const uint32_t w1 = pack_bf16_rne(sc[1][i - 1], sc[1][i]);
                    pn[0][ks2][(i & 7) >> 1] = w0;
                    pn[1][ks2][(i & 7) >> 1] = w1;
                    psum_pair(p0, w0);
                    psum_pair(p1, w1);
                }
#pragma unroll
                for (int j = (i & 7) * NI / 8; j < ((i & 7) + 1) * NI / 8; j++) {
                    if (i < 8) copy_one(src_k, dst_k, j);
                    else copy_one(src_v, dst_v, j);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            ps[0] = p0;
            ps[1] = p1;
        };
        auto issue_copies = [&](int t) {                                 // what step t fetches
            if (t + 3 < n_tiles) issue(Kg, lds_k + (uint32_t)(((t + 3) & 1) * PF_TILE), t + 3);
            if (t + 2 < n_tiles) issue(Vg, lds_v + (uint32_t)(((t + 2) % 3) * PF_TILE), t + 2);
        };

        // prologue (K(0), V(0), K(1), V(1) are on their way), K(2); scores and softmax of tile 0 (sets the reference),
        // scores of tile 1.  From then on step t fetches K(t+3) and V(t+2).
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // K(0), V(0), K(1), V(1)
        PF_LDS_BARRIER();
        u32x4 pa[2][2], pb[2][2], pl[2][2];
        f32x16 sa[2], sb[2];
        scores(0, sa, -1, -1);
#pragma unroll
        for (int c = 0; c < 2; c++) {
            (void)sm_move_ref(c, sm_prep(0, c, sa[c]));                     // nothing accumulated yet
            sm_finish(c, sa[c], pa[c], pl[c]);
        }
        if (n_tiles > 1) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            PF_LDS_BARRIER();
            if (n_tiles > 2) issue(Kg, lds_k, 2);
            scores(1, sa, -1, -1);
        }
        // now: sa = raw scores of tile t+1, pa = weights of tile t, for t = 0
        const int d0 = (int)((first_masked_key + 1) / PF_TK);            // tiles 0 .. d0-1 need no mask
        int t = 0;
        bool slow = false;
        bool top_done = false;                                           // the top of step t has been passed already
        auto more = [&]() -> bool { return t + 1 < d0 && t + 2 < n_tiles; };
        if (more()) {
            step_top();
            fetch(0, 0, 0, 0);
            fetch(0, 0, 1, 1);
            top_done = true;
            for (;;) {
                float ps[2];
                pstep(t, t3, sa, sb, pa, pb, ps);
                if (__any(ps[0] > BIG || ps[1] > BIG)) { slow = true; break; }
                l_part[0] += ps[0];
                l_part[1] += ps[1];
                t++;
                t3 = next3(t3);
                if (!more()) {
                    score_done(sb);
#pragma unroll
                    for (int c = 0; c < 2; c++) {
                        sa[c] = sb[c];
                        pa[c][0] = pb[c][0];
                        pa[c][1] = pb[c][1];
                    }
                    break;
                }
                pstep(t, t3, sb, sa, pb, pa, ps);
                if (__any(ps[0] > BIG || ps[1] > BIG)) { slow = true; break; }
                l_part[0] += ps[0];
                l_part[1] += ps[1];
                t++;
                t3 = next3(t3);
                if (!more()) break;
            }
            score_done(sa);
        }
        // the tiles on the diagonal and the tail, in sequence
        if (!slow)
            for (; t < n_tiles; t++) {
                if (!top_done) step_top();
                top_done = false;
                issue_copies(t);
                bool bad = false;
                const float l_save[2] = {l_part[0], l_part[1]};
                if (t + 1 < n_tiles) {
                    const float x0 = sm_prep(t + 1, 0, sa[0]), x1 = sm_prep(t + 1, 1, sa[1]);
                    sm_finish(0, sa[0], pb[0], pl[0]);
                    sm_finish(1, sa[1], pb[1], pl[1]);
                    bad = __any(x0 > m_ref[0] + SLACK || x1 > m_ref[1] + SLACK);
                }
                values(t, pa, pl);
                if (bad) {
                    l_part[0] = l_save[0];
                    l_part[1] = l_save[1];
                    slow = true;
                    break;
                }
                if (t + 2 < n_tiles) scores(t + 2, sa, -1, -1);
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    pa[c][0] = pb[c][0];
                    pa[c][1] = pb[c][1];
                }
            }
        // slow loop (rare): entered after the top, the copies and the value products of step t; the
        // reference follows the maximum and the accumulators are rescaled every tile
        if (slow) {
            bool resumed = true;
            for (; t + 1 < n_tiles; t++) {
                if (!resumed) {
                    if (!top_done) step_top();
                    top_done = false;
                    issue_copies(t);
                }
                f32x16 s[2];
                scores_global(t + 1, s);
                float corr[2];
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    corr[c] = sm_move_ref(c, sm_prep(t + 1, c, s[c]));
                    sm_finish(c, s[c], pb[c], pl[c]);
                }
                if (!resumed) values(t, pa, pl);
                resumed = false;
                rescale(corr);
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    pa[c][0] = pb[c][0];
                    pa[c][1] = pb[c][1];
                }
            }
            if (!top_done) step_top();
            values(n_tiles - 1, pa, pl);
        }
    }

    // ---- epilogue ----
    if constexpr (SPLIT) {
        float *part = slice->part, *part_ml = slice->part_ml;
        if (part) {
            // a slice's share, in the order the registers hold it: every store is one KiB
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const float l = l_part[c] + __shfl_xor(l_part[c], 32, 64);
                if (g == 0) *(f32x2 *)(part_ml + ((wave * 2 + c) * 32 + l32) * 2) = (f32x2){m_ref[c], l};
#pragma unroll
                for (int db = 0; db < 8; db++)
#pragma unroll
                    for (int b4 = 0; b4 < 4; b4++) {
                        f32x4 w;
#pragma unroll
                        for (int i = 0; i < 4; i++) w[i] = oacc[c][db][4 * b4 + i];
                        *(f32x4 *)(part + ((((wave * 2 + c) * 8 + db) * 4 + b4) * 64 + lane) * 4) = w;
                    }
            }
            return;
        }
    }
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const float inv = pf_reciprocal(l_part[c] + __shfl_xor(l_part[c], 32, 64), m_ref[c]);
        const int r = wave * 64 + 32 * c + l32;
        if (t0 + r % P < n) {
            float *o = out + (t0 + r % P) * q_stride + (size_t)(kvh * GROUP + r / P) * PF_HD + 4 * g;
#pragma unroll
            for (int db = 0; db < 8; db++)
#pragma unroll
                for (int b4 = 0; b4 < 4; b4++) {
                    f32x4 w;
#pragma unroll
                    for (int i = 0; i < 4; i++) w[i] = oacc[c][db][4 * b4 + i] * inv;
                    *(f32x4 *)(o + 32 * db + 8 * b4) = w;
                }
        }
    }
}

// the last workgroup to leave puts the counters back to zero for the next launch (every
// workgroup has drawn its last ticket before it counts itself out)
__device__ __forceinline__ void pf_tickets_done(uint32_t *__restrict__ tickets) {
    if (threadIdx.x == 0) {
        const uint32_t gone = atomicAdd(&tickets[1], 1u);
        if (gone == gridDim.x - 1) {
            __hip_atomic_store(&tickets[0], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&tickets[1], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

template <int GROUP, int WAVES>
__host__ __device__ inline int64_t pf_block_keys(int64_t pos0, int64_t n, int64_t pblk) {
    return pf_keys(pos0, n, 64 * WAVES / GROUP, pblk);
}

// One launch: position blocks below n_prec take the PRECISE body.
template <int GROUP>
__global__ void __launch_bounds__(64 * PF_WAVES, 1)
gqa_prefill_kernel(const uint16_t *__restrict__ K, const uint16_t *__restrict__ V,
                   const uint16_t *__restrict__ Q, int64_t pos0, int64_t n, int n_kv_heads,
                   float scale_log2e, float *__restrict__ out, int64_t n_prec, int64_t pblocks,
                   uint32_t *__restrict__ tickets) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    __shared__ uint32_t sh_item;
    // One workgroup per compute unit stays for the whole launch and draws its (position block,
    // kv head) items from a counter: a compute unit that the dispatcher would leave empty for
    // 4 to 30 us between two workgroups goes on at once, and XCDs that run slower than the others
    // (two of the eight took 6 % longer for the same share) simply draw fewer items.  Items are
    // handed out from the most expensive position block to the cheapest (the last ones to start
    // must be the short ones).  A block costs its number of key tiles, and 1.6 times that in the
    // PRECISE variant: rank r = item / n_kv_heads in the merge of the two descending sequences
    // 10 (p+1), p >= n_prec, and 16 (p+1), p < n_prec.
    // The first item of a workgroup is its own index, without a ticket: read-modify-writes of one
    // address from all XCDs are served one after the other (about 0.15 us each), so a first
    // draw by every workgroup at once would start the last of them tens of microseconds late.
    // Later draws come one by one as the items end.
    const uint32_t total = (uint32_t)(pblocks * n_kv_heads);
    uint32_t item = blockIdx.x;
    for (;;) {
        if (item >= total) break;
        const int64_t rank = (int64_t)item / n_kv_heads;
        // (a scalar for good: the division leaves it in a vector register, and what the copies' addresses are made of with it)
        uint32_t kvh = item % (uint32_t)n_kv_heads;
        asm volatile("" : "+s"(kvh));
        int64_t pblk = -1, before = 0;                  // precise blocks ranked before this one
        for (int64_t pp = n_prec - 1; pp >= 0; pp--) {
            int64_t qmin = 16 * (pp + 1) / 10;          // plain blocks q >= qmin cost more than precise block pp
            if (qmin < n_prec) qmin = n_prec;
            const int64_t rk = (qmin < pblocks ? pblocks - qmin : 0) + (n_prec - 1 - pp);
            if (rk == rank) pblk = pp;
            if (rk < rank) before++;
        }
        if (pblk < 0) pblk = pblocks - 1 - (rank - before);
        const int64_t keys = pf_block_keys<GROUP, PF_WAVES>(pos0, n, pblk);
        if (pblk < n_prec) gqa_prefill_body<GROUP, true, false>(smem_raw, K, V, Q, pos0, n, keys, n_kv_heads, scale_log2e, out, pblk, (int)kvh);
        else gqa_prefill_body<GROUP, false, false>(smem_raw, K, V, Q, pos0, n, keys, n_kv_heads, scale_log2e, out, pblk, (int)kvh);
        // nothing of the last item may still be on its way into LDS
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (threadIdx.x == 0) sh_item = gridDim.x + atomicAdd(&tickets[0], 1u);
        __syncthreads();
        item = __builtin_amdgcn_readfirstlane(sh_item);
        __syncthreads();                                 // everybody has the item, and is done with the last one's LDS
    }
    pf_tickets_done(tickets);
}

// What the first loads of a workgroup need comes in the arguments that arrive in registers; the plan, which whole blocks
// do without, is searched through the scalar cache (2 900 cycles from a kernel's first instruction to its first load; in
// one trip of a vector load, eight entries a lane: 3 % slower).
struct PfWork {
    int kvh, rank, slice, n_slices;
};
__device__ __forceinline__ PfWork pf_work(uint32_t item, uint32_t n_kv_heads, int pblocks, int per, const PfPlan &plan) {
    uint32_t slice_no;
    if (n_kv_heads & (n_kv_heads - 1)) slice_no = item / n_kv_heads;
    else slice_no = item >> __builtin_ctz(n_kv_heads);
    PfWork w = {(int)(item - slice_no * n_kv_heads), (int)slice_no, 0, 1};
    if (!per) return w;
    int lo = 0, hi = pblocks;                           // the rank with first[rank] <= slice_no < first[rank + 1]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if ((uint32_t)plan.first[mid] <= slice_no) lo = mid;
        else hi = mid;
    }
    w.rank = lo;
    w.slice = (int)slice_no - plan.first[lo];
    w.n_slices = plan.first[lo + 1] - plan.first[lo];
    return w;
}

// The same for chunks whose position blocks do not fill the chip: a block's keys are dealt to several
// workgroups, each with whole tiles, and gqa_prefill_merge_kernel combines what they leave.
// What it costs is the partials: 256 KB written and read per slice of 256 rows, 252 slices of 34 tiles
// for 517 positions behind 7083 on four kv heads.  That chunk took 310 us on its 36 workgroups and takes
// 90 (with the preparation of its rows).  (Partials by non-temporal stores: 3 us slower.)
template <int WAVES> constexpr size_t PF_PART = (size_t)64 * WAVES * PF_HD;     // floats of one slice's accumulators

template <int GROUP>
__global__ void __launch_bounds__(64 * PF_WAVES, 1)
gqa_prefill_split_kernel(const uint16_t *__restrict__ K, const uint16_t *__restrict__ V,
                         const uint16_t *__restrict__ Q, int pos0_, int n_, uint32_t n_kv_heads_, int pblocks, int per, int n_prec,
                         float scale_log2e,
                         // (up to here they arrive in registers)
                         float *__restrict__ out, const PfPlan plan, float *__restrict__ part, float *__restrict__ part_ml,
                         uint32_t *__restrict__ tickets) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    __shared__ uint32_t sh_item;
    __shared__ PfSlice sh_slice;
    const int64_t pos0 = pos0_, n = n_;
    const int n_kv_heads = (int)n_kv_heads_;
    uint32_t item = blockIdx.x;                         // (no more workgroups than items)
    for (;;) {
        const PfWork w = pf_work(item, n_kv_heads_, pblocks, per, plan);
        const int kvh = w.kvh, slice = w.slice, n_slices = w.n_slices;
        const int64_t pblk = pblocks - 1 - w.rank;
        const int64_t k0 = (int64_t)slice * per * PF_TK;
        int64_t keys = pf_block_keys<GROUP, PF_WAVES>(pos0, n, pblk) - k0;
        if (slice + 1 < n_slices) keys = (int64_t)per * PF_TK;
        const size_t row0 = (size_t)k0 * n_kv_heads * PF_HD;
        // (read behind the body's barriers; the last item's reads are behind the draw's)
        if (threadIdx.x == 0) sh_slice = {n_slices > 1 ? part + item * PF_PART<PF_WAVES> : nullptr, part_ml + (size_t)item * (64 * PF_WAVES * 2)};
        if (pblk < n_prec)
            gqa_prefill_body<GROUP, true, true>(smem_raw, K + row0, V + row0, Q, pos0 - k0, n, keys, n_kv_heads,
                                                scale_log2e, out, pblk, kvh, &sh_slice);
        else
            gqa_prefill_body<GROUP, false, true>(smem_raw, K + row0, V + row0, Q, pos0 - k0, n, keys, n_kv_heads,
                                                 scale_log2e, out, pblk, kvh, &sh_slice);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const uint32_t total = (uint32_t)(per ? (int)plan.first[pblocks] : pblocks) * n_kv_heads_;
        if (gridDim.x >= total) return;                  // one item each: nothing to draw
        if (threadIdx.x == 0) sh_item = gridDim.x + atomicAdd(&tickets[0], 1u);
        __syncthreads();
        item = __builtin_amdgcn_readfirstlane(sh_item);
        __syncthreads();
        if (item >= total) break;
    }
    pf_tickets_done(tickets);
}

// ---- workgroups whose four waves share one block of 64 rows ----
// For problems of few rows or few keys.  What 256 rows cost besides their tiles (18 us: query rows, first
// tiles, the tiles at either end of the pipeline in sequence, 256 KB of output) and what slices of them leave
// behind (256 KB of partials each, written and read) is most of such a problem's time.  Here a wave takes every
// fourth key tile of the same 64 rows, copies it into its own part of LDS and works on it alone, without
// barriers; the four meet in LDS at the end.  A tile serves 64 rows instead of 256: a step of four tiles takes
// 1.65 us, 2.1 with every compute unit at it (2048 cycles of it matrix instructions), and what is in the way is
// the copies.  One buffer each for K and V: K(u + 1) is on its way during the softmax and the value products of
// tile u, V(u + 1) during the next scores.
// Calls replayed from a graph, in the best plan of workgroups of 256 rows and as they are dealt, those of few steps to the
// other body: 1000 positions of 16 heads on 4 kv heads 47.0 and 31.3 us, 360 29.9 and 17.3, 100 20.6 and 10.0, 16 11.7 and 7.7;
// 1000 of 8 / 8 43.7 and 25.4; 2500 of 16 98.1 and 80.5; 29 behind 3219 31.8 and 15.8, 128 of 8 / 8 behind 1800 29.4 and 14.9,
// 16 behind 16000 43.3 and 24.0.  Long chunks go the other way: 517 behind 7083 take 109 us in the best plan of such workgroups,
// 84.7 in workgroups of 256 rows.
// One copy global -> LDS: 16 bytes a lane from a scalar base and the lane's offset, to a scalar place and a constant beyond it.
// (The constant is added inside: outside, sixteen places a tile are sixteen scalars that live through the loops, more than
// there are, and go in and out of lanes of vector registers.  With this and the arguments in registers: 16 positions of 16
// heads 6.94 -> 6.61 us, 100 9.67 -> 9.10, 64 of 16 / 2 8.99 -> 8.39, 1500 44.1 -> 42.3, 2500 of 16 / 4 85.1 -> 82.2.)
#define PF_COPY(off, base, place, by)                                                                                    \
    do {                                                                                                                 \
        uint32_t at_;                                                                                                    \
        asm volatile("s_add_u32 %0, %3, %4\n\ts_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"              \
                     : "=&s"(at_) : "v"(off), "s"(base), "s"(place), "n"(by) : "memory", "scc");                         \
    } while (0)
struct PfTeamSmem {
    unsigned char k[PF_WAVES][PF_TILE], v[PF_WAVES][PF_TILE];   // at the end: the accumulators that change hands
    unsigned char q[PF_TILE];                                   // query rows 32 .. 63 (block B)
    f32x2 ml[PF_WAVES][64];                                     // a wave's reference and weight sum of every row
};

// For more than PF_ROUNDS2 or PF_ROUNDS steps of four tiles (gqa_prefill_rounds_body has the others): every wave has tiles.
static_assert(PF_ROUNDS >= 1 && PF_ROUNDS2 >= 1, "a wave without a tile");
template <int GROUP, bool PRECISE>
__device__ __forceinline__ void
gqa_prefill_team_body(unsigned char *smem_raw, const uint16_t *__restrict__ K, const uint16_t *__restrict__ V,
                      const uint16_t *__restrict__ Q, int64_t pos0, int64_t n, int64_t wg_keys, int n_kv_heads,
                      float scale_log2e, float *__restrict__ out, int64_t pblk, int kvh, float *part, float *part_ml) {
    constexpr int P = 64 / GROUP;           // positions per workgroup
    constexpr int NI = 16;                  // copies of a tile
    PfTeamSmem &sm = *reinterpret_cast<PfTeamSmem *>(smem_raw);
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));           // (see gqa_prefill_body)
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31;
    const int g = lane >> 5;                // 0/1

    const int64_t t0 = pblk * P;
    const int n_heads = n_kv_heads * GROUP;
    const int64_t q_stride = (int64_t)n_heads * PF_HD;
    const int n_tiles = (int)((wg_keys + PF_TK - 1) / PF_TK);
    const int my_tiles = (n_tiles - wave + PF_WAVES - 1) / PF_WAVES;        // tiles wave, wave + 4, ...
    const int64_t first_masked_key = pos0 + t0;

    const uint32_t row_bytes = (uint32_t)n_kv_heads * (PF_HD * 2);
    uint32_t cp_off = (uint32_t)(16 * g) * row_bytes + (uint32_t)l32 * 16;
    asm volatile("" : "+v"(cp_off));
    const unsigned char *Kg = (const unsigned char *)(K + (size_t)kvh * PF_HD);
    const unsigned char *Vg = (const unsigned char *)(V + (size_t)kvh * PF_HD);
    const uint32_t lds_k = (uint32_t)(uintptr_t)(pf_lds_void *)&sm.k[wave][0];
    const uint32_t lds_v = (uint32_t)(uintptr_t)(pf_lds_void *)&sm.v[wave][0];
    // copy i of a tile takes rows i and i + 16 (gqa_prefill_body's copies)
    auto issue = [&](const unsigned char *base, uint32_t lds_tile, int tile) {
        const uint32_t key0 = (uint32_t)tile * PF_TK;
        const uint32_t left = (uint32_t)wg_keys - 1 - key0;
        const uint64_t first = (uint64_t)base + (uint64_t)key0 * row_bytes;
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)first), hi = __builtin_amdgcn_readfirstlane((uint32_t)(first >> 32));
        const unsigned char *src = (const unsigned char *)((uint64_t)hi << 32 | lo);
        const uint32_t last = (left < PF_TK ? left : PF_TK - 1) * row_bytes + (PF_HD * 2 - 16);
#pragma unroll
        for (int i = 0; i < NI; i++) {
            uint32_t off = (i >= 8 ? cp_off ^ 16 : cp_off) + (uint32_t)i * row_bytes;
            off = off < last ? off : last;
            PF_COPY(off, src, lds_tile, i * PF_PAIR);
        }
    };

    // Query rows, sixteen pairs of rows of either block, dealt to the waves; block A goes through the last
    // wave's V buffer on its way into fragments.  The first tiles are requested with them.
    {
        const int c = wave >> 1;
        const uint32_t lds_q = (uint32_t)(uintptr_t)(pf_lds_void *)(c ? &sm.q[0] : &sm.v[PF_WAVES - 1][0]);
        const int64_t left = n - 1 - t0;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int m = 8 * (wave & 1) + j;
            const int r = 32 * c + m + 16 * g;
            const uint32_t t = (uint32_t)(r % P) < left ? (uint32_t)(r % P) : (uint32_t)left;
            const uint32_t off = t * ((uint32_t)n_heads * (PF_HD * 2)) + (uint32_t)(r / P) * (PF_HD * 2) + ((uint32_t)l32 ^ pf_swap(m)) * 16;
            PF_COPY(off, Q + t0 * q_stride + (size_t)kvh * GROUP * PF_HD, lds_q + (uint32_t)(8 * (wave & 1) * PF_PAIR), j * PF_PAIR);
        }
    }
    issue(Kg, lds_k, wave);
    if (wave != PF_WAVES - 1) issue(Vg, lds_v, wave);
    f32x16 oacc[2][8];
    auto clear = [&]() {
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int db = 0; db < 8; db++) {
#pragma unroll
                for (int i = 0; i < 16; i++) oacc[c][db][i] = 0.0f;
                asm volatile("" : "+a"(oacc[c][db]));
            }
    };
    clear();                                // (while the copies are on their way)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    PF_LDS_BARRIER();
    bf16x8 qf[16];
    {
        const unsigned char *a = &sm.v[PF_WAVES - 1][pf_row(l32) + ((g ^ pf_swap(l32)) << 4)];
#pragma unroll
        for (int ks = 0; ks < 16; ks++) qf[ks] = __builtin_bit_cast(bf16x8, *(const u32x4 *)(a + 32 * ks));
    }
    PF_LDS_BARRIER();
    if (wave == PF_WAVES - 1) issue(Vg, lds_v, wave);

    const unsigned char *kfrag = &sm.k[wave][pf_row(l32) + ((g ^ pf_swap(l32)) << 4)];
    const unsigned char *qfrag = &sm.q[pf_row(l32) + ((g ^ pf_swap(l32)) << 4)];
    const int grp = lane >> 4, gi = lane & 15;
    const int v_key0 = 4 * (grp >> 1) + (gi >> 2);
    const int v_col = 2 * (grp & 1) + ((gi & 3) >> 1);
    const unsigned char *vfrag[2] = {&sm.v[wave][pf_row(v_key0) + (v_col << 4) + (gi & 1) * 8],
                                     &sm.v[wave][pf_row(v_key0 + 8) + ((v_col ^ 1) << 4) + (gi & 1) * 8]};
    auto vread = [&](int st, int half) -> s16x4 {
        return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(vfrag[half] + (st & 7) * 64 + (st >> 3) * 512));
    };

    float m_ref[2] = {-INFINITY, -INFINITY}, l_part[2] = {0.0f, 0.0f};

    auto scores = [&](f32x16 (&s)[2]) {
        u32x4 ka[PF_PRE], qa[PF_PRE];
#pragma unroll
        for (int ks = 0; ks < PF_PRE; ks++) {
            ka[ks] = *(const u32x4 *)(kfrag + 32 * ks);
            qa[ks] = *(const u32x4 *)(qfrag + 32 * ks);
        }
#pragma unroll
        for (int ks = 0; ks < 16; ks++) {
            const bf16x8 kf = __builtin_bit_cast(bf16x8, ka[ks % PF_PRE]);
            const bf16x8 q1 = __builtin_bit_cast(bf16x8, qa[ks % PF_PRE]);
            if (ks + PF_PRE < 16) {
                ka[ks % PF_PRE] = *(const u32x4 *)(kfrag + 32 * (ks + PF_PRE));
                qa[ks % PF_PRE] = *(const u32x4 *)(qfrag + 32 * (ks + PF_PRE));
            }
            if (ks == 0) {
                asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(s[0]) : "v"(kf), "v"(qf[ks]));
                asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(s[1]) : "v"(kf), "v"(q1));
            } else {
                asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(s[0]) : "v"(kf), "v"(qf[ks]));
                asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(s[1]) : "v"(kf), "v"(q1));
            }
        }
        // (the wait carries the scores: without, nothing keeps the first instruction that reads them behind it)
        asm volatile("s_nop 15\n\ts_nop 15" : "+v"(s[0]), "+v"(s[1])::"memory");
    };
    // masks the raw scores of a tile and returns this lane's maximum in log2 units
    auto prep = [&](int tile, int c, f32x16 &s) -> float {
        const int64_t key0 = (int64_t)tile * PF_TK;
        float tmax = -INFINITY;
        if (key0 + PF_TK - 1 > first_masked_key) {
            const int left = (int)(n - 1 - t0 < P ? n - 1 - t0 : P), tr = (32 * c + l32) % P;
            const int lim = (int)(first_masked_key - key0) + (tr < left ? tr : left) - 4 * g;
#pragma unroll
            for (int i = 0; i < 16; i++)
                if ((i >> 2) * 8 + (i & 3) > lim) s[i] = -INFINITY;
        }
#pragma unroll
        for (int i = 0; i < 16; i++) tmax = fmaxf(tmax, s[i]);
        return tmax * scale_log2e;
    };
    auto finish = [&](int c, f32x16 &s, u32x4 (&pw)[2], u32x4 (&pl)[2]) {
        const float m_use = m_ref[c] == -INFINITY ? 0.0f : m_ref[c];
        float psum = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            s[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], scale_log2e, -m_use));
            if (PRECISE) psum += s[i];
        }
#pragma unroll
        for (int ks2 = 0; ks2 < 2; ks2++)
#pragma unroll
            for (int h = 0; h < 4; h++) {
                pw[ks2][h] = pack_bf16_rne(s[8 * ks2 + 2 * h], s[8 * ks2 + 2 * h + 1]);
                if (PRECISE)
                    pl[ks2][h] = pack_bf16_rne(s[8 * ks2 + 2 * h] - bf16lo_to_f32(pw[ks2][h]),
                                               s[8 * ks2 + 2 * h + 1] - bf16hi_to_f32(pw[ks2][h]));
                else
                    psum = pair_sum_bf16(pw[ks2][h], psum);
            }
        l_part[c] += psum;
    };
    constexpr float SLACK = 64.0f;
    auto move_ref = [&](int c, float tmax) -> float {
        tmax = xor32_max(tmax);
        float corr = 1.0f;
        if (tmax > m_ref[c] + 8.0f) {
            corr = __builtin_amdgcn_exp2f(m_ref[c] - tmax);
            m_ref[c] = tmax;
            l_part[c] *= corr;
        }
        return corr;
    };
    // (the accumulators pinned to AGPRs: left to the allocator, some of them change sides in every tile)
    auto value_mfma = [&](f32x16 &acc, bf16x8 a, const u32x4 &b) {
        asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
    };
    auto values = [&](u32x4 (&pw)[2][2], u32x4 (&pl)[2][2]) {
        s16x4 lo[PF_PRE], hi[PF_PRE];
#pragma unroll
        for (int st = 0; st < PF_PRE; st++) lo[st] = vread(st, 0), hi[st] = vread(st, 1);
        // all weights are in their registers, two wait states in front of the first product
        if (PRECISE) asm volatile("" : "+v"(pl[0][0]), "+v"(pl[0][1]), "+v"(pl[1][0]), "+v"(pl[1][1]));
        asm volatile("s_nop 1" : "+v"(pw[0][0]), "+v"(pw[0][1]), "+v"(pw[1][0]), "+v"(pw[1][1])::"memory");
#pragma unroll
        for (int st = 0; st < 16; st++) {
            const int ks2 = st >> 3, db = st & 7;
            typedef __attribute__((ext_vector_type(8))) short s16x8;
            const bf16x8 va = __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(lo[st % PF_PRE], hi[st % PF_PRE], 0, 1, 2, 3, 4, 5, 6, 7));
            if (st + PF_PRE < 16) lo[st % PF_PRE] = vread(st + PF_PRE, 0), hi[st % PF_PRE] = vread(st + PF_PRE, 1);
            value_mfma(oacc[0][db], va, pw[0][ks2]);
            value_mfma(oacc[1][db], va, pw[1][ks2]);
            if (PRECISE) {
                value_mfma(oacc[0][db], va, pl[0][ks2]);
                value_mfma(oacc[1][db], va, pl[1][ks2]);
            }
        }
    };
    auto values_done = [&]() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); };     // before a VALU read of the accumulators
    auto rescale = [&](const float (&corr)[2]) {            // in place (see gqa_prefill_body)
        values_done();
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int db = 0; db < 8; db++)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    float tmp;
                    asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\ts_nop 0\n\t"
                                 "v_accvgpr_write_b32 %0, %1"
                                 : "+a"(oacc[c][db][i]), "=&v"(tmp)
                                 : "v"(corr[c]));
                }
    };
    // The oldest tile in flight has landed: behind it the copies of at most one other are on their way.
    auto landed = [&](bool other) {
        if (other) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NI) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };
    // the fragments of a buffer have been read: its next tile may come
    auto next_tile = [&](const unsigned char *base, uint32_t lds_tile, int u) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (u < my_tiles) issue(base, lds_tile, wave + PF_WAVES * u);
    };

    // All of the wave's tiles.  FOLLOW: the reference follows the maximum and the accumulators are rescaled every
    // tile; without, the reference stays at the first tile's maximum, and a tile with a row that outgrew it ends the
    // attempt (false).  (A row whose keys of a tile are all masked sees nothing of later tiles either: every row
    // has its reference from the first tile.)
    auto tiles = [&](auto follow) -> bool {
        constexpr bool FOLLOW = decltype(follow)::value;
        for (int u = 0;;) {
            f32x16 s[2];
            u32x4 pw[2][2], pl[2][2];
            landed(true);
            scores(s);
            next_tile(Kg, lds_k, u + 1);
            const int tile = wave + PF_WAVES * u;
            const float x[2] = {prep(tile, 0, s[0]), prep(tile, 1, s[1])};
            if constexpr (FOLLOW) {
                const float corr[2] = {move_ref(0, x[0]), move_ref(1, x[1])};
                rescale(corr);
            } else if (__any(x[0] > m_ref[0] + SLACK || x[1] > m_ref[1] + SLACK)) {
                if (u > 0) return false;
                (void)move_ref(0, x[0]);                    // nothing accumulated yet
                (void)move_ref(1, x[1]);
            }
            finish(0, s[0], pw[0], pl[0]);
            finish(1, s[1], pw[1], pl[1]);
            landed(u + 1 < my_tiles);
            values(pw, pl);
            next_tile(Vg, lds_v, u + 1);
            if (++u == my_tiles) return true;
        }
    };
    if (!tiles(std::false_type{})) {
        // a row outgrew its reference (rare): from the first tile again
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");
        clear();
        m_ref[0] = m_ref[1] = -INFINITY;
        l_part[0] = l_part[1] = 0.0f;
        issue(Kg, lds_k, wave);
        issue(Vg, lds_v, wave);
        (void)tiles(std::true_type{});
    }

    // ---- the waves meet: a quarter of the dims at a time, in two places of LDS in turn; of a quarter's sixteen
    // pieces (a column block, 32 dims, 8 of them) a wave adds up those of one column block and 32 dims ----
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const float l = xor32_sum(l_part[c]);
        if (g == 0) sm.ml[wave][32 * c + l32] = (f32x2){m_ref[c], l};
    }
    values_done();
    PF_LDS_BARRIER();                                       // (and all waves are done with their tiles)
    const int cw = wave >> 1, dw = wave & 1, r = 32 * cw + l32;
    float f[2], top = 0.0f, sum = 0.0f;
#pragma unroll
    for (int c = 0; c < 2; c++) {
        f32x2 ml[PF_WAVES];
        float t = -INFINITY, l = 0.0f;
#pragma unroll
        for (int w = 0; w < PF_WAVES; w++) {
            ml[w] = sm.ml[w][32 * c + l32];
            t = fmaxf(t, ml[w][0]);
        }
#pragma unroll
        for (int w = 0; w < PF_WAVES; w++)
            if (ml[w][0] > -INFINITY) l = __builtin_fmaf(ml[w][1], __builtin_amdgcn_exp2f(ml[w][0] - t), l);
        f[c] = m_ref[c] > -INFINITY ? __builtin_amdgcn_exp2f(m_ref[c] - t) : 0.0f;
        if (c == cw) top = t, sum = l;
    }
    const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
    const bool row = t0 + r % P < n;
    float *o = out + (t0 + r % P) * q_stride + (size_t)(kvh * GROUP + r / P) * PF_HD + 32 * dw + 4 * g;
    float *po = part + ((cw * 8 + dw) * 4 * 64 + lane) * 4;
    f32x4 *put = (f32x4 *)smem_raw + wave * 16 * 64 + lane;
    const f32x4 *get = (const f32x4 *)smem_raw + (cw * 2 + dw) * 4 * 64 + lane;
#pragma unroll
    for (int qd = 0; qd < 4; qd++) {
        const int place = PF_WAVES * (qd & 1) * 16 * 64;
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int d = 0; d < 2; d++)
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    f32x4 w;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        float x;
                        asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x) : "a"(oacc[c][2 * qd + d][4 * b + i]));
                        w[i] = x * f[c];
                    }
                    put[place + ((c * 2 + d) * 4 + b) * 64] = w;
                }
        PF_LDS_BARRIER();
        f32x4 w[4];
#pragma unroll
        for (int b = 0; b < 4; b++) w[b] = get[place + b * 64];
#pragma unroll
        for (int v = 1; v < PF_WAVES; v++)
#pragma unroll
            for (int b = 0; b < 4; b++) w[b] += get[place + (v * 16 + b) * 64];
#pragma unroll
        for (int b = 0; b < 4; b++) {
            if (part) *(f32x4 *)(po + (2 * qd * 4 + b) * 256) = w[b];
            else if (row) *(f32x4 *)(o + 64 * qd + 8 * b) = w[b] * inv;
        }
    }
    if (part && dw == 0 && g == 0) *(f32x2 *)(part_ml + r * 2) = (f32x2){top, sum};
}

// The same for workgroups of few steps (PF_ROUNDS, PF_ROUNDS2).  Four waves with accumulators of their own clear, and at the
// end meet in, 256 KB of them: 11 500 cycles of the 27 000 of a block of one step, LDS takes 64 bytes of the writes a
// cycle.  Here the waves score a tile each as there, but hand the weights round in LDS, and each accumulates a quarter of the
// dims over all four tiles: nothing meets at the end but the weight sums, and the query's second block has room in
// registers.  For that they go in step, two barriers a round (four with two-term weights, whose LDS has room for one block of
// rows at a time), with one reference for a row; K(u + 1) is copied beside the value products, V(u) beside the scores.  A
// round takes 6 000 cycles (8 300 with two-term weights), a step of the other 4 400 and 5 900: the copies, 500 cycles of
// the compute unit's memory pipeline for a tile, find the other's waves at different places.  (The scores of round u + 1
// beside the softmax of round u as well, out of two sets of score registers: the copies no longer land in time, 1000
// positions 34.1 -> 35.5 us.  The operands of the next tile's products fetched ahead: equal.)
// Replayed from a graph, 16 heads on 4 kv heads: 16 positions 7.9 -> 6.9 us, 100 11.8 -> 9.7, 360 17.9 -> 16.8, 700
// 25.5 -> 24.6; 50 of 8 / 8 10.5 -> 8.3; 200 of 16 / 2 14.8 -> 12.9; 29 behind 3219, with their preparation, 21.4 -> 18.0, 128 of
// 8 / 8 behind 1800 20.3 -> 17.5, 16 behind 16000 27.3 -> 25.5, 300 of 16 / 2 behind 500 28.9 -> 27.1.  For all steps: 1000
// positions 31.8 -> 34.1, 900 behind 3000 79 -> 84.5.
struct PfRoundsSmem {
    unsigned char k[PF_WAVES][PF_TILE], v[PF_WAVES][PF_TILE];
    // query rows 32 .. 63 on their way into registers, then the weights of four tiles: [tile][four fragments][lane]
    union {
        unsigned char q[PF_TILE];
        u32x4 w[PF_WAVES][4][64];
    };
    float top[PF_WAVES][64];                                    // a wave's maximum of every row, at the end its weight sum
    uint32_t outgrown[PF_WAVES];
};
static_assert(sizeof(PfRoundsSmem) <= 160 * 1024 - 64, "LDS");
constexpr size_t PF_TEAM_LDS = sizeof(PfRoundsSmem) > sizeof(PfTeamSmem) ? sizeof(PfRoundsSmem) : sizeof(PfTeamSmem);

template <int GROUP, bool PRECISE>
__device__ __forceinline__ void
gqa_prefill_rounds_body(unsigned char *smem_raw, const uint16_t *__restrict__ K, const uint16_t *__restrict__ V,
                      const uint16_t *__restrict__ Q, int64_t pos0, int64_t n, int64_t wg_keys, int n_kv_heads,
                      float scale_log2e, float *__restrict__ out, int64_t pblk, int kvh, float *part, float *part_ml) {
    constexpr int P = 64 / GROUP;           // positions per workgroup
    constexpr int NI = 16;                  // copies of a tile
    PfRoundsSmem &sm = *reinterpret_cast<PfRoundsSmem *>(smem_raw);
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));           // (see gqa_prefill_body)
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31;
    const int g = lane >> 5;                // 0/1

    const int64_t t0 = pblk * P;
    const int n_heads = n_kv_heads * GROUP;
    const int64_t q_stride = (int64_t)n_heads * PF_HD;
    const int n_tiles = (int)((wg_keys + PF_TK - 1) / PF_TK);
    const int64_t first_masked_key = pos0 + t0;

    const uint32_t row_bytes = (uint32_t)n_kv_heads * (PF_HD * 2);
    uint32_t cp_off = (uint32_t)(16 * g) * row_bytes + (uint32_t)l32 * 16;
    asm volatile("" : "+v"(cp_off));
    const unsigned char *Kg = (const unsigned char *)(K + (size_t)kvh * PF_HD);
    const unsigned char *Vg = (const unsigned char *)(V + (size_t)kvh * PF_HD);
    const uint32_t lds_k = (uint32_t)(uintptr_t)(pf_lds_void *)&sm.k[wave][0];
    const uint32_t lds_v = (uint32_t)(uintptr_t)(pf_lds_void *)&sm.v[wave][0];
    // copy i of a tile takes rows i and i + 16 (gqa_prefill_body's copies)
    struct TileSrc {
        const unsigned char *base;
        uint32_t last;
    };
    auto tile_src = [&](const unsigned char *base, int tile) -> TileSrc {
        const uint32_t key0 = (uint32_t)tile * PF_TK;
        const uint32_t left = (uint32_t)wg_keys - 1 - key0;
        const uint64_t first = (uint64_t)base + (uint64_t)key0 * row_bytes;
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)first), hi = __builtin_amdgcn_readfirstlane((uint32_t)(first >> 32));
        return {(const unsigned char *)((uint64_t)hi << 32 | lo), (left < PF_TK ? left : PF_TK - 1) * row_bytes + (PF_HD * 2 - 16)};
    };
    auto copy_one = [&](const TileSrc &src, uint32_t lds_tile, int i) {
        uint32_t off = (i >= 8 ? cp_off ^ 16 : cp_off) + (uint32_t)i * row_bytes;
        off = off < src.last ? off : src.last;
        PF_COPY(off, src.base, lds_tile, i * PF_PAIR);
    };
    auto issue = [&](const unsigned char *base, uint32_t lds_tile, int tile) {
        const TileSrc src = tile_src(base, tile);
#pragma unroll
        for (int i = 0; i < NI; i++) copy_one(src, lds_tile, i);
    };

    // Query rows, sixteen pairs of rows of either block, dealt to the waves; block A goes through the last
    // wave's V buffer on its way into fragments.  The first tiles are requested with them.
    {
        const int c = wave >> 1;
        const uint32_t lds_q = (uint32_t)(uintptr_t)(pf_lds_void *)(c ? &sm.q[0] : &sm.v[PF_WAVES - 1][0]);
        const int64_t left = n - 1 - t0;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int m = 8 * (wave & 1) + j;
            const int r = 32 * c + m + 16 * g;
            const uint32_t t = (uint32_t)(r % P) < left ? (uint32_t)(r % P) : (uint32_t)left;
            const uint32_t off = t * ((uint32_t)n_heads * (PF_HD * 2)) + (uint32_t)(r / P) * (PF_HD * 2) + ((uint32_t)l32 ^ pf_swap(m)) * 16;
            PF_COPY(off, Q + t0 * q_stride + (size_t)kvh * GROUP * PF_HD, lds_q + (uint32_t)(8 * (wave & 1) * PF_PAIR), j * PF_PAIR);
        }
    }
    const bool single = n_tiles == 1 && !part;
    const int first_tile = single ? 0 : wave;
    if (first_tile < n_tiles) {
        issue(Kg, lds_k, first_tile);
        if (wave != PF_WAVES - 1) issue(Vg, lds_v, first_tile);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    PF_LDS_BARRIER();
    bf16x8 qf[2][16];
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const unsigned char *a = (c ? &sm.q[0] : &sm.v[PF_WAVES - 1][0]) + pf_row(l32) + ((g ^ pf_swap(l32)) << 4);
#pragma unroll
        for (int ks = 0; ks < 16; ks++) qf[c][ks] = __builtin_bit_cast(bf16x8, *(const u32x4 *)(a + 32 * ks));
    }
    PF_LDS_BARRIER();
    if (wave == PF_WAVES - 1 && first_tile < n_tiles) issue(Vg, lds_v, first_tile);

    const unsigned char *kfrag = &sm.k[wave][pf_row(l32) + ((g ^ pf_swap(l32)) << 4)];
    const int grp = lane >> 4, gi = lane & 15;
    const int v_key0 = 4 * (grp >> 1) + (gi >> 2);
    const int v_col = 2 * (grp & 1) + ((gi & 3) >> 1);
    const unsigned char *vfrag[2] = {&sm.v[wave][pf_row(v_key0) + (v_col << 4) + (gi & 1) * 8],
                                     &sm.v[wave][pf_row(v_key0 + 8) + ((v_col ^ 1) << 4) + (gi & 1) * 8]};
    float m_ref[2] = {-INFINITY, -INFINITY}, l_part[2] = {0.0f, 0.0f};

    // after_step(ks) is called behind every pair of products
    auto scores = [&](f32x16 (&s)[2], auto after_step) {
        u32x4 ka[PF_PRE];
#pragma unroll
        for (int ks = 0; ks < PF_PRE; ks++) ka[ks] = *(const u32x4 *)(kfrag + 32 * ks);
#pragma unroll
        for (int ks = 0; ks < 16; ks++) {
            const bf16x8 kf = __builtin_bit_cast(bf16x8, ka[ks % PF_PRE]);
            if (ks + PF_PRE < 16) ka[ks % PF_PRE] = *(const u32x4 *)(kfrag + 32 * (ks + PF_PRE));
            if (ks == 0) {
                asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(s[0]) : "v"(kf), "a"(qf[0][ks]));
                asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(s[1]) : "v"(kf), "a"(qf[1][ks]));
            } else {
                asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(s[0]) : "v"(kf), "a"(qf[0][ks]));
                asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(s[1]) : "v"(kf), "a"(qf[1][ks]));
            }
            after_step(ks);
        }
        // (the wait carries the scores: without, nothing keeps the first instruction that reads them behind it)
        asm volatile("s_nop 15\n\ts_nop 15" : "+v"(s[0]), "+v"(s[1])::"memory");
    };
    // masks the raw scores of a tile and returns this lane's maximum in log2 units
    auto prep = [&](int tile, int c, f32x16 &s) -> float {
        const int64_t key0 = (int64_t)tile * PF_TK;
        float tmax = -INFINITY;
        if (key0 + PF_TK - 1 > first_masked_key) {
            const int left = (int)(n - 1 - t0 < P ? n - 1 - t0 : P), tr = (32 * c + l32) % P;
            const int lim = (int)(first_masked_key - key0) + (tr < left ? tr : left) - 4 * g;
#pragma unroll
            for (int i = 0; i < 16; i++)
                if ((i >> 2) * 8 + (i & 3) > lim) s[i] = -INFINITY;
        }
#pragma unroll
        for (int i = 0; i < 16; i++) tmax = fmaxf(tmax, s[i]);
        return tmax * scale_log2e;
    };
    auto finish = [&](int c, f32x16 &s, u32x4 (&pw)[2], u32x4 (&pl)[2]) {
        const float m_use = m_ref[c] == -INFINITY ? 0.0f : m_ref[c];
        float psum = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            s[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], scale_log2e, -m_use));
            if (PRECISE) psum += s[i];
        }
#pragma unroll
        for (int ks2 = 0; ks2 < 2; ks2++)
#pragma unroll
            for (int h = 0; h < 4; h++) {
                pw[ks2][h] = pack_bf16_rne(s[8 * ks2 + 2 * h], s[8 * ks2 + 2 * h + 1]);
                if (PRECISE)
                    pl[ks2][h] = pack_bf16_rne(s[8 * ks2 + 2 * h] - bf16lo_to_f32(pw[ks2][h]),
                                               s[8 * ks2 + 2 * h + 1] - bf16hi_to_f32(pw[ks2][h]));
                else
                    psum = pair_sum_bf16(pw[ks2][h], psum);
            }
        l_part[c] += psum;
    };
    constexpr float SLACK = 64.0f;
    auto move_ref = [&](int c, float tmax) -> float {
        tmax = xor32_max(tmax);
        float corr = 1.0f;
        if (tmax > m_ref[c] + 8.0f) {
            corr = __builtin_amdgcn_exp2f(m_ref[c] - tmax);
            m_ref[c] = tmax;
            l_part[c] *= corr;
        }
        return corr;
    };
    // A block of one tile: every wave scores it, and takes a quarter of the dims of the value products to the output
    // (16 positions: 11.0 us where one wave took them all, 7.6 so, 6.8 with all that came later).
    if (single) {
        f32x16 s[2], acc[2][2];
        u32x4 pw[2][2], pl[2][2];
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        scores(s, [](int) {});
#pragma unroll
        for (int c = 0; c < 2; c++) {
            (void)move_ref(c, prep(0, c, s[c]));
            finish(c, s[c], pw[c], pl[c]);
#pragma unroll
            for (int d = 0; d < 2; d++)
#pragma unroll
                for (int i = 0; i < 16; i++) acc[c][d][i] = 0.0f;
        }
        typedef __attribute__((ext_vector_type(8))) short s16x8;
#pragma unroll
        for (int st = 0; st < 4; st++) {
            const int ks2 = st >> 1, d = st & 1, off = wave * 128 + d * 64 + ks2 * 512;
            const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(vfrag[0] + off));
            const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(vfrag[1] + off));
            const bf16x8 va = __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
            for (int c = 0; c < 2; c++) {
                acc[c][d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, __builtin_bit_cast(bf16x8, pw[c][ks2]), acc[c][d], 0, 0, 0);
                if (PRECISE)
                    acc[c][d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, __builtin_bit_cast(bf16x8, pl[c][ks2]), acc[c][d], 0, 0, 0);
            }
        }
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const float inv = pf_reciprocal(xor32_sum(l_part[c]), m_ref[c]);
            const int r = 32 * c + l32;
            if (t0 + r % P < n) {
                float *o = out + (t0 + r % P) * q_stride + (size_t)(kvh * GROUP + r / P) * PF_HD + 64 * wave + 4 * g;
#pragma unroll
                for (int d = 0; d < 2; d++)
#pragma unroll
                    for (int b = 0; b < 4; b++) {
                        f32x4 w;
#pragma unroll
                        for (int i = 0; i < 4; i++) w[i] = acc[c][d][4 * b + i] * inv;
                        *(f32x4 *)(o + 32 * d + 8 * b) = w;
                    }
            }
        }
        return;
    }

    // Round by round, four tiles at a time.  FOLLOW: the reference follows the maximum and the accumulators are rescaled
    // every round; without, the reference stays at the first round's maximum, and a round with a row that outgrew it ends the
    // attempt of all waves (false).  (A row whose keys of a tile are all masked sees nothing of later tiles either: every row
    // has its reference from the first round.)
    f32x16 oacc[2][2];                                      // rows of block c, dims 64 wave + 32 d ..
    // The wait behind the value products carries the accumulators: the compiler moves them about as well, where a loop
    // around the rescaling takes them out of the accumulation registers.
    auto values_done = [&]() {
        asm volatile("s_nop 15\n\ts_nop 15" : "+a"(oacc[0][0]), "+a"(oacc[0][1]), "+a"(oacc[1][0]), "+a"(oacc[1][1])::"memory");
    };
    const int rounds = (n_tiles + PF_WAVES - 1) / PF_WAVES;
    const unsigned char *vquarter[2] = {vfrag[0] - wave * (PF_TILE - 128), vfrag[1] - wave * (PF_TILE - 128)};     // of tile 0
    auto tiles = [&](auto follow) -> bool {
        constexpr bool FOLLOW = decltype(follow)::value;
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int d = 0; d < 2; d++)
#pragma unroll
                for (int i = 0; i < 16; i++) asm volatile("v_accvgpr_write_b32 %0, 0" : "=a"(oacc[c][d][i]));
        for (int u = 0;; u++) {
            const int tile = wave + PF_WAVES * u, here = n_tiles - PF_WAVES * u < PF_WAVES ? n_tiles - PF_WAVES * u : PF_WAVES;
            const bool mine = wave < here, more = tile + PF_WAVES < n_tiles;
            f32x16 s[2];
            u32x4 pw[2][2], pl[2][2];
            float x[2] = {-INFINITY, -INFINITY};
            if (mine) {
                // K(u) has landed; V(u), whose place the round before has left, comes beside the scores
                if (u == 0) {
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NI) : "memory");
                    scores(s, [](int) {});
                } else {
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    const TileSrc src = tile_src(Vg, tile);
                    scores(s, [&](int i) { copy_one(src, lds_v, i); });
                }
                x[0] = prep(tile, 0, s[0]), x[1] = prep(tile, 1, s[1]);
            }
            float corr[2] = {1.0f, 1.0f};
            if (FOLLOW || u == 0) {
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    const float t = xor32_max(x[c]);
                    if (g == 0) sm.top[wave][32 * c + l32] = t;
                }
                PF_LDS_BARRIER();
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    const int r = 32 * c + l32;
                    const float t = fmaxf(fmaxf(sm.top[0][r], sm.top[1][r]), fmaxf(sm.top[2][r], sm.top[3][r]));
                    if (t > m_ref[c] + 8.0f) {
                        corr[c] = __builtin_amdgcn_exp2f(m_ref[c] - t);         // first round: exp2(-inf) = 0
                        m_ref[c] = t;
                        l_part[c] *= corr[c];
                    }
                }
                if (FOLLOW && u > 0) {
#pragma unroll
                    for (int c = 0; c < 2; c++)
#pragma unroll
                        for (int d = 0; d < 2; d++)
#pragma unroll
                            for (int i = 0; i < 16; i++) {          // (in place: see gqa_prefill_body)
                                float tmp;
                                asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\ts_nop 0\n\t"
                                             "v_accvgpr_write_b32 %0, %1"
                                             : "+a"(oacc[c][d][i]), "=&v"(tmp)
                                             : "v"(corr[c]));
                            }
                }
            } else {
                const bool out = __any(x[0] > m_ref[0] + SLACK || x[1] > m_ref[1] + SLACK);
                if (lane == 0) sm.outgrown[wave] = out;
            }
            if (mine) {
                finish(0, s[0], pw[0], pl[0]);
                finish(1, s[1], pw[1], pl[1]);
            }
            // The weights change hands in the order the registers hold them: lane l of every wave reads what lane l wrote.
            // Weights of single precision go all at once, two-term ones a block of rows after the other.
            typedef __attribute__((ext_vector_type(8))) short s16x8;
            const TileSrc next_k = tile_src(Kg, more ? tile + PF_WAVES : 0);
            auto values = [&](int j, int first_c) {         // tile j of the round; beside the first two K(u + 1) comes
                u32x4 w[4];
                bf16x8 va[2][2];                            // [16 keys][32 dims]
#pragma unroll
                for (int f = 0; f < 4; f++) w[f] = sm.w[j][f][lane];
#pragma unroll
                for (int ks2 = 0; ks2 < 2; ks2++)
#pragma unroll
                    for (int d = 0; d < 2; d++) {
                        const int off = j * PF_TILE + d * 64 + ks2 * 512;
                        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(vquarter[0] + off));
                        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(vquarter[1] + off));
                        va[ks2][d] = __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                    }
#pragma unroll
                for (int f = 0; f < 4; f++) {
                    const int c = PRECISE ? first_c : f >> 1;
#pragma unroll
                    for (int d = 0; d < 2; d++)
                        asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(oacc[c][d]) : "v"(va[f & 1][d]), "v"(w[f]));
                    if (j < 2 && (!PRECISE || first_c == 0) && more) {
                        copy_one(next_k, lds_k, 8 * j + 2 * f);
                        copy_one(next_k, lds_k, 8 * j + 2 * f + 1);
                    }
                }
            };
            if (mine) {
#pragma unroll
                for (int f = 0; f < 4; f++) sm.w[wave][f][lane] = PRECISE ? (f < 2 ? pw[0][f & 1] : pl[0][f & 1]) : pw[f >> 1][f & 1];
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // V(u) has landed
            }
            PF_LDS_BARRIER();
            if (!FOLLOW && u > 0) {
                const u32x4 o = *(const u32x4 *)sm.outgrown;
                if (__builtin_amdgcn_readfirstlane(o[0] | o[1] | o[2] | o[3])) return false;
            }
            auto all_values = [&](int c) {
#pragma unroll
                for (int j = 0; j < PF_WAVES; j++)
                    if (j < here) values(j, c);
            };
            all_values(0);
            if (PRECISE) {
                PF_LDS_BARRIER();
                if (mine)
#pragma unroll
                    for (int f = 0; f < 4; f++) sm.w[wave][f][lane] = f < 2 ? pw[1][f & 1] : pl[1][f & 1];
                PF_LDS_BARRIER();
                all_values(1);
            }
            if (FOLLOW) values_done();
            if (u + 1 == rounds) return true;
            PF_LDS_BARRIER();                               // everybody is done with the round's values and weights
        }
    };
    if (!tiles(std::false_type{})) {
        // a row outgrew its reference (rare): from the first tile again
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        PF_LDS_BARRIER();
        m_ref[0] = m_ref[1] = -INFINITY;
        l_part[0] = l_part[1] = 0.0f;
        if (wave < n_tiles) {
            issue(Kg, lds_k, wave);
            issue(Vg, lds_v, wave);
        }
        (void)tiles(std::true_type{});
    }

    // ---- the waves' sums meet; a wave has all that there is of its 64 dims ----
    values_done();
    PF_LDS_BARRIER();
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const float l = xor32_sum(l_part[c]);
        if (g == 0) sm.top[wave][32 * c + l32] = l;
    }
    PF_LDS_BARRIER();
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const int r = 32 * c + l32;
        const float l = (sm.top[0][r] + sm.top[1][r]) + (sm.top[2][r] + sm.top[3][r]);
        if (part) {
            float *po = part + ((c * 8 + 2 * wave) * 4 * 64 + lane) * 4;
#pragma unroll
            for (int d = 0; d < 2; d++)
#pragma unroll
                for (int b = 0; b < 4; b++)
                    *(f32x4 *)(po + (d * 4 + b) * 256) = (f32x4){oacc[c][d][4 * b], oacc[c][d][4 * b + 1], oacc[c][d][4 * b + 2], oacc[c][d][4 * b + 3]};
            if (wave == c && g == 0) *(f32x2 *)(part_ml + r * 2) = (f32x2){m_ref[c], l};
        } else if (t0 + r % P < n) {
            const float inv = pf_reciprocal(l, m_ref[c]);
            float *o = out + (t0 + r % P) * q_stride + (size_t)(kvh * GROUP + r / P) * PF_HD + 64 * wave + 4 * g;
#pragma unroll
            for (int d = 0; d < 2; d++)
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    f32x4 w;
#pragma unroll
                    for (int i = 0; i < 4; i++) w[i] = oacc[c][d][4 * b + i] * inv;
                    *(f32x4 *)(o + 32 * d + 8 * b) = w;
                }
        }
    }
}

template <int GROUP>
__global__ void __launch_bounds__(64 * PF_WAVES, 1)
gqa_prefill_team_kernel(const uint16_t *__restrict__ K, const uint16_t *__restrict__ V,
                         const uint16_t *__restrict__ Q, int pos0_, int n_, uint32_t n_kv_heads_, int pblocks, int per, int n_prec,
                         float scale_log2e,
                         // (up to here they arrive in registers)
                         float *__restrict__ out, const PfPlan plan, float *__restrict__ part, float *__restrict__ part_ml,
                         uint32_t *__restrict__ tickets) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    __shared__ uint32_t sh_item;
    const int64_t pos0 = pos0_, n = n_;
    const int n_kv_heads = (int)n_kv_heads_;
    uint32_t item = blockIdx.x;                         // (no more workgroups than items)
    for (;;) {
        const PfWork w = pf_work(item, n_kv_heads_, pblocks, per, plan);
        const int kvh = w.kvh, slice = w.slice, n_slices = w.n_slices;
        const int64_t pblk = pblocks - 1 - w.rank;
        const int64_t k0 = (int64_t)slice * per * PF_TK;
        int64_t keys = pf_block_keys<GROUP, 1>(pos0, n, pblk) - k0;
        if (slice + 1 < n_slices) keys = (int64_t)per * PF_TK;
        const size_t row0 = (size_t)k0 * n_kv_heads * PF_HD;
        float *p = n_slices > 1 ? part + item * PF_PART<1> : nullptr, *pml = part_ml + (size_t)item * (64 * 2);
        auto body = [&](auto f) { f(smem_raw, K + row0, V + row0, Q, pos0 - k0, n, keys, n_kv_heads, scale_log2e, out, pblk, kvh, p, pml); };
        if (pblk < n_prec) {
            if (keys <= PF_ROUNDS2 * PF_WAVES * PF_TK) body([](auto... a) { gqa_prefill_rounds_body<GROUP, true>(a...); });
            else body([](auto... a) { gqa_prefill_team_body<GROUP, true>(a...); });
        } else {
            if (keys <= PF_ROUNDS * PF_WAVES * PF_TK) body([](auto... a) { gqa_prefill_rounds_body<GROUP, false>(a...); });
            else body([](auto... a) { gqa_prefill_team_body<GROUP, false>(a...); });
        }
        const uint32_t total = (uint32_t)(per ? (int)plan.first[pblocks] : pblocks) * n_kv_heads_;
        if (gridDim.x >= total) return;                  // one item each: nothing to draw
        if (threadIdx.x == 0) sh_item = gridDim.x + atomicAdd(&tickets[0], 1u);
        __syncthreads();
        item = __builtin_amdgcn_readfirstlane(sh_item);
        __syncthreads();
        if (item >= total) break;
    }
    pf_tickets_done(tickets);
}

// Combines the slices of a block: out = sum_s 2^(m_s - M) acc_s / sum_s 2^(m_s - M) l_s.  A wave
// takes 32 rows x 8 dims (one KiB of the partials per slice, one load), a workgroup a 32-dim output block.
// What it waits for is the partials' way from memory, so the loads of BATCH slices are in flight at once and
// few rows make many waves: 16 positions behind 16000 on four kv heads (64 slices) took 46.6 us, with their
// preparation, of which this kernel had 17, and 32.3 so (a wave for four times the dims, four slices at a time, before).  Blocks of up
// to eight slices are shorter with eight (2500 positions 103 us against 108): the registers of sixteen cost
// waves.
template <int GROUP, int WAVES, int BATCH>
__global__ void __launch_bounds__(256)
gqa_prefill_merge_kernel(const float *__restrict__ part, const float *__restrict__ part_ml, int64_t n,
                         int n_kv_heads, int pblocks, const PfPlan plan, float *__restrict__ out) {
    constexpr int P = 64 * WAVES / GROUP;
    const int rank = blockIdx.x / n_kv_heads, kvh = blockIdx.x % n_kv_heads;
    const int n_slices = plan.first[rank + 1] - plan.first[rank];
    if (n_slices < 2) return;                           // its workgroup wrote the output
    const int cb = blockIdx.y >> 3, db = blockIdx.y & 7;        // column block: 32 rows; output block: 32 dims
    const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
    const int b4 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const size_t item0 = (size_t)plan.first[rank] * n_kv_heads + kvh, step = n_kv_heads;
    const float *ml = part_ml + item0 * (64 * WAVES * 2) + (cb * 32 + l32) * 2;
    const float *pa = part + item0 * PF_PART<WAVES> + ((size_t)((cb * 8 + db) * 4 + b4) * 64 + lane) * 4;
    float mx = -INFINITY, l = 0.0f;
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int s0 = 0; s0 < n_slices; s0 += BATCH) {
        f32x2 v[BATCH];
        f32x4 a[BATCH];
        float top = mx;
#pragma unroll
        for (int j = 0; j < BATCH; j++) {
            v[j] = (f32x2){-INFINITY, 0.0f};
            a[j] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
            if (s0 + j < n_slices) {
                v[j] = *(const f32x2 *)(ml + (s0 + j) * step * (64 * WAVES * 2));
                a[j] = *(const f32x4 *)(pa + (s0 + j) * step * PF_PART<WAVES>);
            }
        }
#pragma unroll
        for (int j = 0; j < BATCH; j++) top = fmaxf(top, v[j][0]);
        const float keep = __builtin_amdgcn_exp2f(mx - top);    // the first slices: exp2(-inf) = 0
        mx = top;
        l *= keep;
        acc *= keep;
#pragma unroll
        for (int j = 0; j < BATCH; j++) {
            const float c = __builtin_amdgcn_exp2f(v[j][0] - mx);
            l = __builtin_fmaf(v[j][1], c, l);
#pragma unroll
            for (int i = 0; i < 4; i++) acc[i] = __builtin_fmaf(a[j][i], c, acc[i]);
        }
    }
    const int r = cb * 32 + l32;
    const int64_t t = (int64_t)(pblocks - 1 - rank) * P + r % P;
    if (t >= n) return;
    *(f32x4 *)(out + (t * n_kv_heads * GROUP + kvh * GROUP + r / P) * PF_HD + 32 * db + 8 * b4 + 4 * g) = acc * (l > 0.0f ? 1.0f / l : 0.0f);
}

// Position blocks that take the PRECISE body: those whose rows see at most this many keys.  Short
// prefixes: few keys carry the whole weight, so the 2^-9 rounding of each bf16 weight shows in an O(1)
// output; the rounding residual through the matrix core as well makes weights good to 2^-17.
static int64_t gqa_precise_keys() {
    static const int64_t v = [] {
        const char *e = getenv("CWICK_HIP_GQA_PRECISE_KEYS");
        const int64_t x = e ? atoll(e) : 1024;
        return x < 0 ? (int64_t)0 : x;
    }();
    return v;
}
template <int GROUP, int WAVES>
static int64_t pf_precise_blocks(int64_t pos0, int64_t n, int64_t pblocks) {
    int64_t n_prec = 0;
    while (n_prec < pblocks && pf_block_keys<GROUP, WAVES>(pos0, n, n_prec) <= gqa_precise_keys()) n_prec++;
    return n_prec;
}

// the dynamic LDS a kernel asks for is allowed once
template <auto KERNEL>
static hipError_t pf_allow_lds(size_t bytes) {
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [&] {
        err = hipFuncSetAttribute((const void *)KERNEL, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    });
    return err;
}

template <int GROUP>
static int run_gqa_prefill_team(const uint16_t *k, const uint16_t *v, int64_t pos0, int64_t n, int n_kv_heads, const uint16_t *q,
                                float scale, float *out, int64_t n_prec, int pblocks, const PfPlan &plan, float *part,
                                uint32_t *tickets, hipStream_t s) {
    CWICK_HIP_CALL((pf_allow_lds<gqa_prefill_team_kernel<GROUP>>(PF_TEAM_LDS)));
    const int slices = plan.first[pblocks] * n_kv_heads;
    float *part_ml = part ? part + (size_t)slices * PF_PART<1> : nullptr;
    {
        ProfKernel pk(CWICK_HIP_PROF_GQA_PREFILL, s);
        pk.launch(gqa_prefill_team_kernel<GROUP>, dim3((unsigned)(slices < num_cus() ? slices : num_cus())), dim3(64 * PF_WAVES),
                  PF_TEAM_LDS, k, v, q, (int)pos0, (int)n, (uint32_t)n_kv_heads, pblocks, plan.per, (int)n_prec, scale * 1.44269504088896340736f, out,
                  plan, part, part_ml, tickets);
    }
    CWICK_HIP_CALL(hipGetLastError());
    if (!plan.per) return 1;
    const bool many = plan.first[1] > 8;                // (no block has more slices than the last)
    (many ? gqa_prefill_merge_kernel<GROUP, 1, 16> : gqa_prefill_merge_kernel<GROUP, 1, 8>)<<<
        dim3((unsigned)(pblocks * n_kv_heads), 16), 256, 0, s>>>(part, part_ml, n, n_kv_heads, pblocks, plan, out);
    CWICK_HIP_CALL(hipGetLastError());
    return 1;
}

template <int GROUP>
static int run_gqa_prefill_split(const uint16_t *k, const uint16_t *v, int64_t pos0, int64_t n, int n_kv_heads, const uint16_t *q,
                                 float scale, float *out, int64_t n_prec, int pblocks, const PfPlan &plan, float *part,
                                 uint32_t *tickets, hipStream_t s) {
    CWICK_HIP_CALL((pf_allow_lds<gqa_prefill_split_kernel<GROUP>>(sizeof(PfSmem))));
    const int slices = plan.first[pblocks] * n_kv_heads;
    float *part_ml = part ? part + (size_t)slices * PF_PART<PF_WAVES> : nullptr;
    {
        ProfKernel pk(CWICK_HIP_PROF_GQA_PREFILL, s);
        pk.launch(gqa_prefill_split_kernel<GROUP>, dim3((unsigned)(slices < num_cus() ? slices : num_cus())), dim3(64 * PF_WAVES),
                  sizeof(PfSmem), k, v, q, (int)pos0, (int)n, (uint32_t)n_kv_heads, pblocks, plan.per, (int)n_prec, scale * 1.44269504088896340736f, out,
                  plan, part, part_ml, tickets);
    }
    CWICK_HIP_CALL(hipGetLastError());
    if (!plan.per) return 1;
    const bool many = plan.first[1] > 8;                // (no block has more slices than the last)
    (many ? gqa_prefill_merge_kernel<GROUP, PF_WAVES, 16> : gqa_prefill_merge_kernel<GROUP, PF_WAVES, 8>)<<<
        dim3((unsigned)(pblocks * n_kv_heads), 16 * PF_WAVES), 256, 0, s>>>(part, part_ml, n, n_kv_heads, pblocks, plan, out);
    CWICK_HIP_CALL(hipGetLastError());
    return 1;
}

// The partials of a plan that cuts blocks.  Null where there is no room for them (a stream that is being captured
// and has not run the shape before): the blocks then stay whole.
template <int WAVES>
static float *pf_partials(const PfPlan &plan, int pblocks, int n_kv_heads, hipStream_t s) {
    const size_t slices = (size_t)plan.first[pblocks] * n_kv_heads;
    return (float *)workspace_if_free(s, slices * (PF_PART<WAVES> + 64 * WAVES * 2) * sizeof(float));
}

template <int GROUP>
static int run_gqa_prefill(const uint16_t *k, const uint16_t *v, int64_t pos0, int64_t n,
                           int n_kv_heads, const uint16_t *q, float scale, float *out,
                           hipStream_t s) {
    constexpr int P = 64 * PF_WAVES / GROUP;
    const int64_t pblocks = (n + P - 1) / P, items = pblocks * n_kv_heads;
    CWICK_REQUIRE(items <= 0x7FFFFFFF, "gqa_prefill: grid too large");
    const int64_t n_prec = pf_precise_blocks<GROUP, PF_WAVES>(pos0, n, pblocks);
    uint32_t *tickets = ticket_counters(s);
    if (!tickets) return 0;                 // ticket_counters() has recorded why
    // From two items per compute unit on the tickets even the blocks out; below that some units
    // would have one item, or none.  The plans of both ways to deal the chunk are priced, and a plan that
    // cuts blocks needs room for the partials.
    PfPlan plan, team_plan;
    constexpr int TEAM_P = 64 / GROUP;
    const int64_t team_blocks = (n + TEAM_P - 1) / TEAM_P, team_prec = pf_precise_blocks<GROUP, 1>(pos0, n, team_blocks);
    float t = INFINITY;
    if (items < 2 * num_cus() && pblocks <= PF_MAX_BLOCKS)
        t = pf_plan(pos0, n, P, n_kv_heads, n_prec, num_cus(), PF_COST_WIDE, t, plan);
    else plan.per = 0;
    if (team_blocks <= PF_MAX_BLOCKS && t < INFINITY &&
        pf_plan(pos0, n, TEAM_P, n_kv_heads, team_prec, num_cus(), PF_COST_TEAM, t, team_plan) < t) {
        float *part = team_plan.per ? pf_partials<1>(team_plan, (int)team_blocks, n_kv_heads, s) : nullptr;
        if (part || !team_plan.per)
            return run_gqa_prefill_team<GROUP>(k, v, pos0, n, n_kv_heads, q, scale, out, team_prec, (int)team_blocks, team_plan, part, tickets, s);
    }
    if (float *part = plan.per ? pf_partials<PF_WAVES>(plan, (int)pblocks, n_kv_heads, s) : nullptr)
        return run_gqa_prefill_split<GROUP>(k, v, pos0, n, n_kv_heads, q, scale, out, n_prec, (int)pblocks, plan, part, tickets, s);
    CWICK_HIP_CALL((pf_allow_lds<gqa_prefill_kernel<GROUP>>(sizeof(PfSmem))));
    const int64_t wgs = items < num_cus() ? items : num_cus();      // the LDS of a compute unit holds one workgroup
    {
        ProfKernel pk(CWICK_HIP_PROF_GQA_PREFILL, s);
        pk.launch(gqa_prefill_kernel<GROUP>, dim3((unsigned)wgs), dim3(64 * PF_WAVES), sizeof(PfSmem),
                  k, v, q, pos0, n, n_kv_heads, scale * 1.44269504088896340736f, out, n_prec, pblocks, tickets);
    }
    CWICK_HIP_CALL(hipGetLastError());
    return 1;
}

int launch_gqa_prefill(const uint16_t *k, const uint16_t *v, int64_t pos0, int64_t n,
                       int n_kv_heads, int head_dim, const uint16_t *q, int n_heads, float scale,
                       float *out, hipStream_t s) {
    CWICK_REQUIRE(k && v && q && out, "gqa_prefill: null pointer");
    CWICK_REQUIRE(pos0 >= 0 && n >= 1 && pos0 + n <= ((int64_t)1 << 30),
                  "gqa_prefill: pos0 %lld n %lld", (long long)pos0, (long long)n);
    CWICK_REQUIRE(head_dim == PF_HD, "gqa_prefill: head_dim %d is not supported (256 only)", head_dim);
    CWICK_REQUIRE(n_kv_heads >= 1 && n_heads >= n_kv_heads && n_heads % n_kv_heads == 0,
                  "gqa_prefill: n_heads %d is not a multiple of n_kv_heads %d", n_heads, n_kv_heads);
    CWICK_REQUIRE(scale > 0.0f && scale < INFINITY, "gqa_prefill: scale must be positive");
    CWICK_REQUIRE(((uintptr_t)k | (uintptr_t)v | (uintptr_t)q | (uintptr_t)out) % 16 == 0,
                  "gqa_prefill: K, V, q and out must be 16-byte aligned");
    switch (n_heads / n_kv_heads) {
        case 1: return run_gqa_prefill<1>(k, v, pos0, n, n_kv_heads, q, scale, out, s);
        case 2: return run_gqa_prefill<2>(k, v, pos0, n, n_kv_heads, q, scale, out, s);
        case 4: return run_gqa_prefill<4>(k, v, pos0, n, n_kv_heads, q, scale, out, s);
        case 8: return run_gqa_prefill<8>(k, v, pos0, n, n_kv_heads, q, scale, out, s);
        default: break;
    }
    set_error("gqa_prefill: group %d is not supported (1, 2, 4, 8)", n_heads / n_kv_heads);
    return 0;
}

}  // namespace cwick
