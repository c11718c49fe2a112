// mla_roles.hip -- absorbed-latent MLA over the FP8 latent: decode and sparse decode
// (src/attention.c:749-811).
//
//   workgroup = 12 waves, 32 query rows (heads of one query) x one key slice, walked in tiles
//   of 64 keys.  The waves take one of two roles:
//     waves 0..7  score: wave (kb, hh) takes keys 16 kb..+15 of the tile and heads 16 hh..+15:
//                 S^T = K Q^T on v_mfma_scale_f32_16x16x128_f8f6f4 with K as stored (E4M3) and Q
//                 as two E4M3 terms with a shared E8M0 scale per head and 128-dim block; the five
//                 block products are combined with the keys' fp32 block scales, exponentiated
//                 against the wave's reference m, and published through LDS as fp16
//                 probabilities exp2(s - m), already in the fragment order of the value MFMA,
//                 together with m;
//     waves 8..11 accumulate: wave cw owns output dims 128 cw..+127 (one scale block) for all 32
//                 heads: it turns the probabilities into weights p * scale[key][cw] * 2^(10 - e)
//                 (packed fp16 multiplies; 2^e is above every scale the wave has seen, so the
//                 weights fit fp16) and runs O^T += V^T W^T on v_mfma_f32_16x16x32_f16, V^T read
//                 transposed from the tile (ds_read_b64_tr_b8) and widened E4M3 -> fp16 (exact).
//   The roles are one tile apart (tile t+1 is scored while tile t is accumulated), so a step has
//   a single workgroup barrier and nobody waits for an exchange inside it.  The softmax
//   reference is lazy: a scoring wave keeps the reference every wave knows (m_ref) unless its own
//   tile exceeds it by 2^LAZY; the m it used travels with the probabilities together with one
//   flag per scoring wave ("my reference for this tile is not the common one").  One step later
//   every wave reads the eight flags: all clear (almost always) means nothing to do; otherwise
//   the accumulating waves (and the scorers, for their sums) bring everything to the common
//   maximum.  Each scoring lane keeps the sum of its own keys; the sums meet once, after the loop.
//   Tiles are copied global -> LDS by global_load_lds (no registers) into four stages.  Tiles 0 to 2
//   are fetched by all twelve waves around the preparation of Q; from step 0 on every wave copies its share of
//   tile t+3 during step t (a scoring wave the 512 latent bytes of eight keys, a value wave the rope bytes of
//   sixteen and a scale block): the value waves at the top of the step, the scoring waves at the end of theirs,
//   when they would otherwise wait at the barrier.  The copies are issued from inline assembly and the barrier
//   waits for LDS traffic only, so the compiler never makes anything wait for the tiles in
//   flight.  LDS is addressed by integer byte offsets throughout (a generic pointer into LDS costs
//   a null check and a 64-bit add per use), and the kernel exists in two instantiations: dense
//   lists (rows are k_begin + i, only the last tile can be ragged) and lists given by sel[].
//
//   Where the time goes (cycle stamps, 12 waves on 256 CUs): a 64-key step has 1 088 cycles of matrix work on
//   a SIMD and takes 2 100 to 2 300.  No unit is saturated: the two scoring waves and the value wave of a SIMD are
//   chains of instructions, each of which takes its wave five cycles whatever its kind, of LDS round trips and of
//   products.  So what pays is fewer instructions in the chain and fewer waits in it: the steps with a whole tile
//   to copy have no condition and no 64-bit multiplication in them (running addresses; the step as a function of its
//   kind), everything a step reads is requested before the first product, the keys' scales are two registers
//   out of which the folds take their factor by DPP, eight flags are eight bytes.  32768 rows of 128 heads, the
//   whole call: 25.2 -> 23.5 us, 22.7 with the partial's scale found two values an instruction and its stores
//   on their way early, 21.0 (of 21.6, from a graph) with a tile's values prepared a step ahead.  Before the first step a
//   workgroup takes 7 200 cycles; behind the last, until its partial is written, 4 300 to 5 300, with 256 workgroups 9 200
//   (a layer's 3037 rows of 64 heads, one tile each: 13 100 in all).
//   A copy instruction that has one lane per row touches 64 cache lines and moves a tile into LDS in 3 100 cycles when
//   every compute unit does it, one that walks along the rows in 1 900 (copy-only kernels; a list of rows 3 600 and
//   3 450), hence the tile's layout (see Tile).  With 32 query rows per tile the per-tile work that does not
//   depend on the rows (copies, scale handling, conversions of V) is paid per 1 088 matrix cycles; 64 rows would
//   halve it per flop.  Eight or sixteen waves per workgroup (the same work split differently) were measured
//   and are no faster; nor are other priorities of the two roles.
//
//   Split-K partials are stored per 16 heads in accumulator-fragment order
//   [split][16-head block][dim block][lane][4] (every store 1 KiB contiguous);
//   mla_merge_frag16_kernel reads them in the same order with all loads in flight.
#include "common.hpp"
#include "mla_plan.hpp"

#include <cstdlib>
#include <cstring>
#include <mutex>
#include <type_traits>

namespace cwick {
namespace {

constexpr int KDIM = CWICK_HIP_LATENT_KDIM;   // 576
constexpr int VDIM = CWICK_HIP_LATENT_VDIM;   // 512
constexpr int NBLK = CWICK_HIP_LATENT_NBLK;   // 5
constexpr int THREADS = 768;                  // waves 0..7 score, waves 8..11 accumulate values
constexpr int TK = 64;                        // keys per tile
constexpr int HB = 16;                        // heads per head half (partials are laid out per 16 heads)
constexpr int HW = 32;                        // heads per workgroup
constexpr int NST = 4;                        // tile stages
constexpr int NCOL = KDIM / 16;               // 36 sixteen-byte columns per row
constexpr int NDB = VDIM / 16;                // 32 sixteen-dim output blocks
constexpr float LAZY = 4.0f;                  // the reference moves when a tile exceeds it by 2^LAZY
constexpr int WEXP = 10;                      // fp16 weights are p * scale * 2^(WEXP - e), scale < 2^e
constexpr int E_NONE = -1000;                 // no scale seen yet
// the steps of the loop: before tile 0, with the copy of a whole tile, with whatever there is, behind the last tile
constexpr int FIRST = 0, STEADY_ = 1, TAIL = 2, LAST = 3;

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
typedef __attribute__((ext_vector_type(8))) int i32x8;
typedef __attribute__((ext_vector_type(2))) int i32x2;
typedef __attribute__((ext_vector_type(4))) int i32x4;
typedef __attribute__((address_space(3))) i32x2 lds_i32x2;
typedef __attribute__((address_space(3))) void lds_void;

// What a workgroup's first copies need comes as arguments of its own, which arrive in registers with the
// waves (the first fourteen dwords, and no struct among them: a struct is fetched through the scalar cache,
// which a launch finds cold); the rest comes in this, fetched while the first copies are on their way.
struct Rest {
    int64_t row_bstride, scale_bstride;
    const float *sink;        // per head, natural-log units of the scaled scores, or null
    float *out, *part_ml;
    uint32_t *part_acc;
    float scale;
};
struct Params {
    const uint8_t *rows;
    const float *scales;
    int64_t n_rows;
    const int32_t *sel;
    int64_t n_list;
    const uint16_t *q;
    int nh, nq, n_splits;
    int64_t keys_per_split;   // multiple of TK
    Rest rest;
};

// What a masked position of a tile (past the end of the list, a -1 or out-of-range entry of
// sel[]) is fetched from: a row of zero bytes with zero scales.  Its weight is zero already;
// with zero values and zero scales nothing of any cache row that is not in the list (a NaN
// byte, a scale many binades above the others) can reach the products or the fp16 normaliser.
__device__ __attribute__((aligned(16))) uint8_t g_zero_row[KDIM + 64] = {0};
__device__ __attribute__((aligned(16))) float g_zero_scales[8] = {0.0f};

// A tile is 36 blocks of 1 KiB, each what one copy instruction fetches: block 8 cg + kg is the eight columns of
// sixteen bytes 8 cg .. of the keys 8 kg .. +7, block 32 + kq the four rope columns of the keys 16 kq .. +15.
// Byte of column c of a key in its block: the four columns of a quarter of the row stay together (four neighbouring
// lanes of the copy fetch 64 bytes of it), keys are 64 bytes apart, and within its four columns a key takes places
// that depend on which four of the sixteen it belongs to.  The bytes in flight through LDS at a time are those of
// lanes 0..3, 12..15, 20..23, 24..27 (then the others, then the upper half) of a sixteen-byte read and of 32 lanes of a
// transpose read: the Gray code of the four takes them to different banks in both (3.3 and 2.0 cycles a read; keys in order
// 6.0 and 6.0, the number of the four itself 6.0 and 2.0).
__device__ __forceinline__ uint32_t swap_of(uint32_t key) { return ((key >> 2) ^ (key >> 3 & 1)) & 3; }
__device__ __forceinline__ uint32_t place(uint32_t c, uint32_t key, uint32_t keys) {          // keys: of the block, 8 or 16
    return 512 * (c >> 2) + 64 * (key & (keys - 1)) + 16 * ((c & 3) ^ swap_of(key));
}
struct Tile {
    uint8_t kv[NCOL][1024];
    float sc[NBLK][TK];           // [block][key]                   1280 B
    uint32_t valid[2];            // list kernels: bit k = position k of the tile holds a row
    uint32_t pad[2];
};
struct Xch {                       // what the scoring waves publish per tile
    // fp16 probabilities exp2(s - m), laid out as the B fragments of the value MFMA:
    // [head half][32-key half][slot group g][head n][4 dwords]; contraction slot 8 g + j of a
    // half is key 8 g + j of that half
    uint32_t p[2][2][4][16][4];
    float m[2][16][4];            // [head half][head][key block]: the reference m they are relative to
    uint8_t moved[8];             // per scoring wave: its reference for this tile is not the common one
    uint8_t pad[8];
};
struct Smem {
    Tile tile[NST];
    Xch x[2];
};
// Q of one (head half, 128-dim block), unit u = 5 hh + b: 64 bytes per lane, first as copied from memory,
// then in MFMA operand order: two sixteen-byte pieces of the hi term, two of the lo term (the rope block's
// one register set, hi and lo, in place of its hi term).  Parked in the last tile stage and the exchange
// area, neither in use yet, the scale bytes behind it.
constexpr uint32_t PARK = (NST - 1) * (uint32_t)sizeof(Tile), PARK_UNIT = 4096, PARK_LO = 2048, PARK_SC = PARK + 10 * PARK_UNIT;
static_assert(PARK_SC + 10 * 256 <= sizeof(Smem), "Q park area");
static_assert(sizeof(Tile) * NST + 2 * sizeof(Xch) <= 160 * 1024, "LDS");

__device__ __forceinline__ float pow2i(int e) {
    e = e > 126 ? 126 : (e < -126 ? -126 : e);
    return __builtin_bit_cast(float, (uint32_t)(e + 127) << 23);
}

// both fp16 halves of a dword times f
__device__ __forceinline__ uint32_t scale_f16x2(uint32_t x, float f) {
    const _Float16 h = (_Float16)f;
    const f16x2 r = __builtin_bit_cast(f16x2, x) * (f16x2){h, h};
    return __builtin_bit_cast(uint32_t, r);
}

__device__ __forceinline__ uint32_t mul_f16x2(uint32_t a, uint32_t b) {
    const f16x2 r = __builtin_bit_cast(f16x2, a) * __builtin_bit_cast(f16x2, b);
    return __builtin_bit_cast(uint32_t, r);
}

#define LDS_BARRIER() asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory")

// one instruction per max: the compiler's fmaxf quiets both operands first (a v_max of the
// operand with itself) because it may not assume they are not signalling NaNs
__device__ __forceinline__ float vmax(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float vmax3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
// the maximum over eight neighbouring lanes
__device__ __forceinline__ uint32_t lanes8_max(uint32_t v) {
    auto meet = [&](uint32_t o) { v = o > v ? o : v; };
    meet(dpp_u32<0xB1, 0xF>(v));                          // quad_perm [1, 0, 3, 2]
    meet(dpp_u32<0x4E, 0xF>(v));                          // quad_perm [2, 3, 0, 1]
    meet(dpp_u32<0x141, 0xF>(v));                         // row_half_mirror
    return v;
}
// max(|a|, |b|, |c|), NaN if any of them is one
__device__ __forceinline__ float maximum3_abs(float a, float b, float c) {
    float r;
    asm("v_maximum3_f32 %0, |%1|, |%2|, |%3|" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) u32x2 lds_u32x2;
typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
typedef __attribute__((address_space(3))) f32x2 lds_f32x2;
typedef __attribute__((address_space(3))) float lds_f32;
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef __attribute__((address_space(3))) uint8_t lds_u8;
// LDS is addressed by byte offsets held in ordinary integers (a generic pointer into LDS costs a
// null check and a 64-bit add at every use)
#define LDS_AT(type, a) (*(type *)(size_t)(uint32_t)(a))

// LDS offsets of the parts of Smem
constexpr uint32_t TILE_B = sizeof(Tile);
constexpr uint32_t SC_OFF = NCOL * TK * 16;                       // Tile::sc
constexpr uint32_t VALID_OFF = SC_OFF + NBLK * TK * 4;            // Tile::valid
constexpr uint32_t X_OFF = NST * TILE_B;                          // Smem::x
constexpr uint32_t XCH_B = sizeof(Xch);
constexpr uint32_t XM_OFF = 2 * 2 * 4 * 16 * 4 * 4;               // Xch::m
constexpr uint32_t XF_OFF = XM_OFF + 2 * 16 * 4 * 4;              // Xch::moved

// shape: the heads of a query in the low eight bits, the splits above.  splits_inv: 2^31 / splits, rounded up.
// eighth: an eighth of the workgroups, 0 if they are no multiple of eight.
template <bool SEL>
__global__ void __launch_bounds__(THREADS)
mla_roles_kernel(const uint16_t *__restrict__ q, const uint8_t *__restrict__ all_rows, const float *__restrict__ all_scales,
                 const int32_t *__restrict__ all_sel, uint32_t n_list, uint32_t n_rows, uint32_t keys_per_split, uint32_t shape,
                 uint32_t splits_inv, uint32_t eighth, const Rest p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    Smem &sm = *reinterpret_cast<Smem *>(smem_raw);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void *)smem_raw;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool scorer = wave < 8;
    const int kb = wave & 3;         // scoring role: keys 16 kb .. 16 kb + 15 of the tile
    const int hh = (wave >> 2) & 1;  //               heads 16 hh .. 16 hh + 15
    const int cw = wave & 3;         // value role: dims 128 cw .. +127 = scale block cw
    const int n = lane & 15;         // head column / key row of a 16-block / dim row
    const int g = lane >> 4;         // 32-wide contraction block (QK) / 8-wide (PV)

    const int nh = (int)(shape & 255u), n_splits = (int)(shape >> 8);
    // Workgroups go to the eight XCDs round robin: an XCD takes a contiguous eighth of the units (the
    // head blocks of a slice, the slices of a query: what they share stays in one L2).
    // (divisions by multiplication: each is thirty instructions in front of the first load otherwise)
    uint32_t unit = blockIdx.x;
    if (eighth) unit = (unit & 7) * eighth + unit / 8;
    const uint32_t n_hb = (uint32_t)(nh + HW - 1) / HW;                    // one to four: 2^31 / n_hb, rounded up, without a table
    const uint32_t slice = div_by(unit, n_hb == 3 ? 0x2AAAAAABu : 0x80000000u >> (n_hb >> 1)), y = div_by(slice, splits_inv);
    const int hb = (int)(unit - slice * n_hb), split = (int)(slice - y * (uint32_t)n_splits);

    const uint8_t *rows = all_rows;
    const float *scales = all_scales;
    if (y) {                                               // (the first query waits for nothing)
        rows += (size_t)y * p.row_bstride;
        scales += (size_t)y * p.scale_bstride;
    }
    const int32_t *sel = SEL ? all_sel + (size_t)y * n_list : nullptr;
    const uint32_t k_begin = (uint32_t)split * keys_per_split;             // below n_list
    const uint32_t left = n_list - k_begin;
    const int n_keys = (int)(left < keys_per_split ? left : keys_per_split);     // of this workgroup
    const int n_tiles = (n_keys + TK - 1) / TK;

    // The zero row and its scales: where masked positions of a tile are fetched from.  The
    // addresses are taken once, here: inside the loops every mention would be a load from the
    // global offset table.
    uint64_t zrow = (uint64_t)(uintptr_t)g_zero_row, zsc = (uint64_t)(uintptr_t)g_zero_scales;
    asm volatile("" : "+s"(zrow), "+s"(zsc));

    // the row of the cache behind position k of tile t, or -1
    auto row_of = [&](int t, int k) -> int {
        const int i = t * TK + k;
        if (!SEL) return (t < n_tiles && i < n_keys) ? (int)(k_begin + i) : -1;    // rows fit 31 bits (checked by the launcher)
        int r = -1;
        if (t < n_tiles && i < n_keys) {
            r = sel[k_begin + i];
            if ((uint32_t)r >= n_rows) r = -1;
        }
        return r;
    };
    // global -> LDS copies in assembly: the compiler keeps no account of them, so nothing in the
    // loop waits for the tile in flight except the s_waitcnt before the barrier.  Each statement
    // writes M0 itself right before the copy that reads it.  M0 is a reserved register to the
    // compiler (it cannot be named as clobbered); what keeps this safe is that nothing else in
    // this file makes the compiler use M0, which tests/test_mfma_wait_states.py checks on the
    // compiled code.
    auto dma16 = [&](uint64_t gp, uint32_t lds_off) {
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(gp), "s"(lds_off) : "memory");
    };
    auto dma4 = [&](uint64_t gp, uint32_t lds_off) {
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(gp), "s"(lds_off) : "memory");
    };
    auto row_ptr = [&](int r) -> uint64_t { return r >= 0 ? (uint64_t)(uintptr_t)rows + (uint64_t)(uint32_t)r * KDIM : zrow; };
    auto sc_ptr = [&](int r) -> uint64_t { return r >= 0 ? (uint64_t)(uintptr_t)scales + (uint64_t)(uint32_t)r * (NBLK * 4) : zsc; };
    // which of the 64 positions of the tile hold a row (the scoring waves mask the others)
    auto mark = [&](int r, uint32_t tile_off) {
        const uint64_t v = __ballot(r >= 0);
        LDS_AT(lds_u32x2, tile_off + VALID_OFF) = (u32x2){(uint32_t)v, (uint32_t)(v >> 32)};
    };
    // A wave's share of a tile.  Scoring wave w: the blocks of keys 8 w .. +7, lane l key (l / 4) % 8 and column
    // 4 (l / 32) + .. of each of the four.  Value wave cw: the rope block of keys 16 cw .. +15, lane l key l / 4, and
    // the scales of dim block cw (the first one: of the rope block too), lane = key.
    const int key_of = scorer ? 8 * wave + ((lane >> 2) & 7) : 16 * cw + (lane >> 2);
    const uint32_t col_of = (scorer ? (uint32_t)(4 * (lane >> 5)) : 32u) + ((uint32_t)(lane & 3) ^ swap_of(key_of));
    const uint32_t lane_row = (uint32_t)key_of * KDIM + 16u * col_of, lane_sc = (uint32_t)lane * (NBLK * 4);
    // rk: the row of the lane's key, rl: of key `lane` (value waves); whole: a dense tile without a masked position,
    // whose place is a scalar
    struct RowPair { int k, l; };
    // (128 cg bytes to the source are the instruction's immediate offset, which the hardware also adds to the LDS
    // address: M0 is set that much below the block)
#define CWICK_ROLES_BLK(cg, ...) asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, " __VA_ARGS__ " offset:128*" #cg
    auto copy_whole = [&](uint64_t rp, uint64_t sp, uint32_t tile_off) {
        if (scorer) {
            const uint32_t blk = tile_off + (uint32_t)wave * 1024;
#define CWICK_ROLES_COPY(cg) CWICK_ROLES_BLK(cg, "%2") ::"v"(lane_row), "s"(blk + (8 * 1024 - 128) * cg), "s"(rp) : "memory")
            CWICK_ROLES_COPY(0); CWICK_ROLES_COPY(1); CWICK_ROLES_COPY(2); CWICK_ROLES_COPY(3);
#undef CWICK_ROLES_COPY
        } else {
            const uint32_t rope = tile_off + (32u + (uint32_t)cw) * 1024, sc = tile_off + SC_OFF + (uint32_t)cw * (TK * 4);
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2" ::"v"(lane_row), "s"(rope), "s"(rp) : "memory");
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, %2" ::"v"(lane_sc), "s"(sc), "s"(sp + 4 * cw) : "memory");
            if (cw == 0)
                asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, %2" ::"v"(lane_sc), "s"(sc + 4 * (TK * 4)), "s"(sp + 16) : "memory");
        }
    };
    auto share = [&](int t, RowPair r, uint32_t tile_off) {
        if (!SEL && (t + 1) * TK <= n_keys) {
            copy_whole((uint64_t)(uintptr_t)rows + (uint64_t)(k_begin + (uint32_t)t * TK) * KDIM,
                       (uint64_t)(uintptr_t)scales + (uint64_t)(k_begin + (uint32_t)t * TK) * (NBLK * 4), tile_off);
        } else if (scorer) {
            const uint32_t blk = tile_off + (uint32_t)wave * 1024;
            const uint64_t rp = row_ptr(r.k) + 16 * col_of;
#define CWICK_ROLES_COPY(cg) CWICK_ROLES_BLK(cg, "off") ::"v"(rp), "s"(blk + (8 * 1024 - 128) * cg) : "memory")
            CWICK_ROLES_COPY(0); CWICK_ROLES_COPY(1); CWICK_ROLES_COPY(2); CWICK_ROLES_COPY(3);
#undef CWICK_ROLES_COPY
        } else {
            const uint32_t rope = tile_off + (32u + (uint32_t)cw) * 1024, sc = tile_off + SC_OFF + (uint32_t)cw * (TK * 4);
            const uint64_t sp = sc_ptr(r.l);
            dma16(row_ptr(r.k) + 16 * col_of, rope);
            dma4(sp + 4 * cw, sc);
            if (cw == 0) dma4(sp + 16, sc + 4 * (TK * 4));
            if (SEL && cw == 0) mark(r.l, tile_off);
        }
    };
#undef CWICK_ROLES_BLK
    // The same in the steps t < n_steady, in which tile t+3 is whole (dense: a running address; a list: entries
    // without a look at its end).
    const int n_steady = n_keys / TK - 3;
    uint64_t next_rows = (uint64_t)(uintptr_t)rows + (uint64_t)(k_begin + 3 * TK) * KDIM, next_sc = (uint64_t)(uintptr_t)scales + (uint64_t)(k_begin + 3 * TK) * (NBLK * 4);
    auto list_row = [&](int t, int k) -> int {
        const int r = sel[k_begin + (uint32_t)(t * TK + k)];
        return (uint32_t)r < n_rows ? r : -1;
    };
    auto share_steady = [&](int t, RowPair r, uint32_t tile_off) {
        if (SEL) {
            share(t, r, tile_off);
            return;
        }
        copy_whole(next_rows, next_sc, tile_off);
        next_rows += TK * KDIM;
        next_sc += TK * NBLK * 4;
    };
    // copies of a wave's share
#define CWICK_ROLES_WAIT(extra_s, extra_v, extra_v0)                                         \
    do {                                                                                     \
        if (scorer) asm volatile("s_waitcnt vmcnt(" #extra_s ")" ::: "memory");               \
        else if (cw) asm volatile("s_waitcnt vmcnt(" #extra_v ")" ::: "memory");              \
        else asm volatile("s_waitcnt vmcnt(" #extra_v0 ")" ::: "memory");                     \
    } while (0)
    // What comes first.  A copy takes the memory pipeline a cycle for every 64 bytes of a row that it touches.  The
    // query, whose preparation the first barrier waits for, goes along its rows (ten to sixteen lines per instruction; a
    // head's 256 bytes of a unit in sixteen pieces, piece x of head h at place x ^ h, so that the heads of a fragment
    // read come from different banks); then tile 0; tiles 1 and 2 when the wave has converted its unit.  From step 0
    // on tile t+3 is fetched during step t.  The loads of the list entries are in assembly like the copies, so that
    // the wait for them leaves the query in flight.
    int entry_k[3], entry_l[3];
    if (SEL) {                                        // (a workgroup has at least one key)
        auto list_at = [&](int t, int k) -> const int32_t * {
            const int i = t * TK + k;
            return sel + k_begin + (i < n_keys ? i : 0);
        };
        asm volatile("global_load_dword %0, %6, off\n\tglobal_load_dword %1, %7, off\n\tglobal_load_dword %2, %8, off\n\t"
                     "global_load_dword %3, %9, off\n\tglobal_load_dword %4, %10, off\n\tglobal_load_dword %5, %11, off"
                     : "=&v"(entry_k[0]), "=&v"(entry_k[1]), "=&v"(entry_k[2]), "=&v"(entry_l[0]), "=&v"(entry_l[1]), "=&v"(entry_l[2])
                     : "v"(list_at(0, key_of)), "v"(list_at(1, key_of)), "v"(list_at(2, key_of)),
                       "v"(list_at(0, lane)), "v"(list_at(1, lane)), "v"(list_at(2, lane)) : "memory");
    }
    // scoring wave (kb, hh): dims 128 kb .. of the head half; value wave: the rope dims of heads 8 cw .. of the 32, eight dims a lane
    const uint32_t unit_lds = lds0 + PARK + (uint32_t)(5 * hh + kb) * PARK_UNIT;
    const uint64_t q_base = (uint64_t)(uintptr_t)(q + (size_t)(y * (uint32_t)nh) * KDIM + 128 * (scorer ? kb : 4));      // (a scalar)
    auto head_off = [&](int h) -> uint32_t { return (uint32_t)(hb * HW + h < nh ? hb * HW + h : nh - 1) * (KDIM * 2); };
    u32x4 rope;
    if (scorer) {
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int h = 4 * c + g;
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2" ::"v"(head_off(16 * hh + h) + (uint32_t)(16 * (n ^ h))),
                         "s"(unit_lds + (uint32_t)c * 1024), "s"(q_base) : "memory");
        }
        if (SEL) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    } else {
        asm volatile("global_load_dwordx4 %0, %1, %2" : "=&v"(rope) : "v"(head_off(8 * cw + (lane >> 3)) + 16u * (uint32_t)(lane & 7)), "s"(q_base) : "memory");
        if (SEL) asm volatile("s_waitcnt vmcnt(1)" ::: "memory");
    }
    if (SEL) asm volatile("" : "+v"(entry_k[0]), "+v"(entry_k[1]), "+v"(entry_k[2]), "+v"(entry_l[0]), "+v"(entry_l[1]), "+v"(entry_l[2])::"memory");
    auto rows_of = [&](int t) -> RowPair { return {row_of(t, key_of), scorer ? -1 : row_of(t, lane)}; };
    auto first_rows = [&](int t) -> RowPair {
        if (!SEL) return rows_of(t);
        auto row = [&](int r, int k) { return t < n_tiles && t * TK + k < n_keys && (uint32_t)r < n_rows ? r : -1; };
        return {row(entry_k[t], key_of), row(entry_l[t], lane)};
    };
    share(0, first_rows(0), lds0);
    // ---- the wave's part of the query as two E4M3 terms with one E8M0 scale per head and block (the hardware pairs the
    // scale of lane (n, g) with k-elements that live in other lanes of the same head, so the four lanes must
    // agree; both terms use it).  Eight dim blocks for eight waves, two a SIMD, and the rope block, half as wide, dealt
    // to the value waves: a SIMD is through with its conversions, 600 cycles of it a dim block, when it has done 2.25.
    CWICK_ROLES_WAIT(4, 2, 3);                            // the share of tile 0 stays in flight
    if (scorer) {
        // lane (n, g) holds head n of the half, dims 128 b + 32 g + [0, 32)
        u32x4 w[4], hi[2], lo[2];
#pragma unroll
        for (int c = 0; c < 4; c++) w[c] = LDS_AT(lds_u32x4, unit_lds + (uint32_t)(n * 256 + (((4 * g + c) ^ n) & 15) * 16));
        const uint32_t unit_byte = q_two_terms(w, hi, lo);
#pragma unroll
        for (int c = 0; c < 2; c++) {
            LDS_AT(lds_u32x4, unit_lds + (uint32_t)(c * 1024 + lane * 16)) = hi[c];
            LDS_AT(lds_u32x4, unit_lds + PARK_LO + (uint32_t)(c * 1024 + lane * 16)) = lo[c];
        }
        LDS_AT(lds_u32, lds0 + PARK_SC + (uint32_t)((5 * hh + kb) * 256 + lane * 4)) = unit_byte;
    } else {
        // the rope block is one register set: lanes g < 2 hold the hi term of dims 512 + 32 g.., lanes g >= 2 the lo term
        // of dims 512 + 32 (g - 2).. (the key side repeats its bytes); eight lanes here hold a head
        asm volatile("" : "+v"(rope)::"memory");
        q_u16x2 m = {};
#pragma unroll
        for (int d = 0; d < 4; d++) m = q_larger(m, rope[d]);
        uint32_t top = m[0] > m[1] ? m[0] : m[1];
        top = lanes8_max(top);
        const uint32_t unit_byte = q_unit(top), h = 8 * (cw & 1) + (uint32_t)(lane >> 3), d8 = (uint32_t)lane & 7;
        u32x2 hi, lo;
#pragma unroll
        for (int d = 0; d < 2; d++) {
            uint32_t a, b;
            q_two_terms(rope[2 * d], rope[2 * d + 1], unit_byte, a, b);
            hi[d] = a, lo[d] = b;
        }
        const uint32_t at = lds0 + PARK + (5 * (uint32_t)(cw >> 1) + 4) * PARK_UNIT + ((d8 >> 1) & 1) * 1024 + ((d8 >> 2) * 16 + h) * 16 + 8 * (d8 & 1);
        LDS_AT(lds_u32x2, at) = hi;
        LDS_AT(lds_u32x2, at + 32 * 16) = lo;
        if (d8 < 4) LDS_AT(lds_u32, lds0 + PARK_SC + (5 * (uint32_t)(cw >> 1) + 4) * 256 + (d8 * 16 + h) * 4) = unit_byte;
    }
    // tile 0 has landed (this wave's share), what comes behind it stays in flight
    if (n_tiles > 2) {
        share(1, first_rows(1), lds0 + TILE_B);
        share(2, first_rows(2), lds0 + 2 * TILE_B);
        CWICK_ROLES_WAIT(8, 4, 6);
    } else if (n_tiles > 1) {
        share(1, first_rows(1), lds0 + TILE_B);
        CWICK_ROLES_WAIT(4, 2, 3);
    } else {
        CWICK_ROLES_WAIT(0, 0, 0);
    }
    LDS_BARRIER();

    const float c0 = p.scale * 1.44269504088896340736f;   // scores in log2 units
    float m_ref[2] = {-INFINITY, -INFINITY};          // of head 16 h2 + n; every wave tracks the same values

    if (scorer) {
        i32x8 qhi[4], qlo[4], qrope;
        int qsc0 = 0, qsc1;                               // scale bytes of blocks 0..3 / of the rope block
        auto park8 = [&](uint32_t a) -> i32x8 {
            const u32x4 x = LDS_AT(lds_u32x4, a), z = LDS_AT(lds_u32x4, a + 1024);
            return (i32x8){(int)x[0], (int)x[1], (int)x[2], (int)x[3], (int)z[0], (int)z[1], (int)z[2], (int)z[3]};
        };
        const uint32_t pq = lds0 + PARK + (uint32_t)(5 * hh) * PARK_UNIT + (uint32_t)lane * 16;
        const uint32_t pc = lds0 + PARK_SC + (uint32_t)(5 * hh * 256 + lane * 4);
#pragma unroll
        for (int b = 0; b < 4; b++) {
            qhi[b] = park8(pq + (uint32_t)b * PARK_UNIT);
            qlo[b] = park8(pq + (uint32_t)b * PARK_UNIT + PARK_LO);
            qsc0 |= (int)(LDS_AT(lds_u32, pc + (uint32_t)b * 256) << (8 * b));
        }
        qrope = park8(pq + 4 * PARK_UNIT);
        qsc1 = (int)LDS_AT(lds_u32, pc + 4 * 256);
        LDS_BARRIER();                                // before copies or weights land in the park area
        // Nothing the compiler has in flight may cross into the loop: its waits would also wait
        // for the copies.
        asm volatile("" : "+v"(qhi[0]), "+v"(qhi[1]), "+v"(qhi[2]), "+v"(qhi[3]), "+v"(qlo[0]), "+v"(qlo[1]), "+v"(qlo[2]), "+v"(qlo[3]), "+v"(qrope), "+v"(qsc0), "+v"(qsc1));

        float l_priv = 0.0f, l_pend = 0.0f;               // sum over this lane's keys (head 16 hh + n), relative to m_ref / to the tile's m_loc
        float mr = -INFINITY;                             // m_ref of this wave's head half
        // per-lane LDS offsets inside a tile: K fragment (key 16 kb + n, columns 8 b + 2 g and, 16 bytes to either side,
        // the next), the rope block's (columns 32 + 2 (g & 1)); the scales of this lane's row of sixteen lanes, place
        // 4 b + i that of dim block b and key 16 kb + 4 g + i (the rope block's by itself)
        const uint32_t k_off = (uint32_t)(2 * kb + (n >> 3)) * 1024 + place(2 * g, n, 8);
        const uint32_t kr_off = (uint32_t)(32 + kb) * 1024 + place(2 * (g & 1), n, 16);
        const uint32_t s_off = SC_OFF + (uint32_t)(((n >> 2) * TK + 16 * kb + 4 * g + (n & 3)) * 4);
        const uint32_t sr_off = SC_OFF + (uint32_t)((4 * TK + 16 * kb + 4 * g + (n & 3)) * 4);
        // where this lane's four probabilities go: keys 16 (kb & 1) + 4 g + i of half kb >> 1
        const uint32_t xp_off = (uint32_t)(((((hh * 2 + (kb >> 1)) * 4 + 2 * (kb & 1) + (g >> 1)) * 16 + n) * 4 + 2 * (g & 1)) * 4);
        const uint32_t xm_off = XM_OFF + (uint32_t)(((hh * 16 + n) * 4 + kb) * 4);
        const uint32_t xmr_off = XM_OFF + (uint32_t)((hh * 16 + n) * 4 * 4);
        const uint32_t xf_off = XF_OFF + (uint32_t)wave;
        const int tail_tile = n_tiles - 1;
        const bool ragged = (n_keys & (TK - 1)) != 0;

        auto step = [&](int t, auto kind) {
            constexpr bool FLAGS = decltype(kind)::value != FIRST, SCORE = decltype(kind)::value != LAST, STEADY = decltype(kind)::value == STEADY_;
            const uint32_t xb = lds0 + X_OFF + (uint32_t)(t & 1) * XCH_B;         // exchange area of tile t
            const bool do_copy = STEADY || (FLAGS && SCORE && t + 3 < n_tiles);
            int r_cp = -1;                                // fetched here (a list entry is a load), used at the end of the step
            if (SEL && do_copy) r_cp = STEADY ? list_row(t + 3, key_of) : row_of(t + 3, key_of);
            u32x2 fl = {0u, 0u};
            if (FLAGS) fl = LDS_AT(lds_u32x2, xb + XF_OFF);
            const uint32_t tb = lds0 + (uint32_t)((t + 1) & (NST - 1)) * TILE_B;
            const uint32_t xn = lds0 + X_OFF + (uint32_t)((t + 1) & 1) * XCH_B;
            f32x4 S;
            if constexpr (SCORE) {
                // ---- scores S^T[key][head] for keys 16 kb.., heads 16 hh.. of tile t+1 ----
                // All that is read is requested first: eight waves read at the same time, and a fragment requested when the
                // one before it is used costs a round trip each (S ready 1 700 cycles behind the barrier that way).
                // The products are in assembly, which the compiler spaces neither from what reads them nor from what writes what
                // they read: the folds stand behind all of them and wait states, and a statement begins with the two wait states
                // between a vector-ALU write (the constant of the scales, wherever the compiler loads it) and a product.
                const uint32_t ka = tb + k_off, kA = tb + (k_off ^ 16u), kr = tb + kr_off, kR = tb + (kr_off ^ 16u);
                u32x4 k0[NBLK], k1[NBLK];
                float r0, r1;
                k0[0] = LDS_AT(lds_u32x4, ka), k1[0] = LDS_AT(lds_u32x4, kA);
                k0[1] = LDS_AT(lds_u32x4, ka + 8192), k1[1] = LDS_AT(lds_u32x4, kA + 8192);
                r0 = LDS_AT(lds_f32, tb + s_off);
                k0[2] = LDS_AT(lds_u32x4, ka + 16384), k1[2] = LDS_AT(lds_u32x4, kA + 16384);
                k0[3] = LDS_AT(lds_u32x4, ka + 24576), k1[3] = LDS_AT(lds_u32x4, kA + 24576);
                k0[4] = LDS_AT(lds_u32x4, kr), k1[4] = LDS_AT(lds_u32x4, kR);
                r1 = LDS_AT(lds_f32, tb + sr_off);
                __builtin_amdgcn_sched_barrier(0);
                auto key = [&](int b) -> i32x8 {
                    return (i32x8){(int)k0[b][0], (int)k0[b][1], (int)k0[b][2], (int)k0[b][3], (int)k1[b][0], (int)k1[b][1], (int)k1[b][2], (int)k1[b][3]};
                };
                const int one_scales = 0x7F7F7F7F;
                f32x4 acc[NBLK];
#define CWICK_ROLES_PAIR(b, SEL_)                                                                                  \
    asm volatile("s_nop 1\n\tv_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, 0, %4, %5 " SEL_ "\n\t"                   \
                 "v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %3, %0, %4, %5 " SEL_                                    \
                 : "=&v"(acc[b]) : "v"(key(b)), "v"(qhi[b]), "v"(qlo[b]), "v"(one_scales), "v"(qsc0))
                // S (+)= product * scale of the key: out of place 4 b + i of the row, inside the multiply-add
                float sum[4];
#define CWICK_ROLES_FOLD(OP, C, i, r, pl, b) asm volatile(OP " %0, %1, %2 row_newbcast:" #pl " row_mask:0xf bank_mask:0xf" : C(sum[i]) : "v"(r), "v"(acc[b][i]))
#define CWICK_ROLES_FOLD4(OP, C, r, p0, p1, p2, p3, b)                                                                                         \
    CWICK_ROLES_FOLD(OP, C, 0, r, p0, b); CWICK_ROLES_FOLD(OP, C, 1, r, p1, b); CWICK_ROLES_FOLD(OP, C, 2, r, p2, b); CWICK_ROLES_FOLD(OP, C, 3, r, p3, b)
                CWICK_ROLES_PAIR(0, "op_sel:[0,0,0] op_sel_hi:[0,0,0]");
                CWICK_ROLES_PAIR(1, "op_sel:[0,1,0] op_sel_hi:[0,0,0]");
                CWICK_ROLES_PAIR(2, "op_sel:[0,0,0] op_sel_hi:[0,1,0]");
                CWICK_ROLES_PAIR(3, "op_sel:[0,1,0] op_sel_hi:[0,1,0]");
                asm volatile("s_nop 1\n\tv_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, 0, %3, %4 op_sel:[0,0,0] op_sel_hi:[0,0,0]"
                             : "=&v"(acc[4]) : "v"(key(4)), "v"(qrope), "v"(one_scales), "v"(qsc1));
                // (fourteen instructions behind the last product of block 0, and more behind the others')
                asm volatile("s_nop 6" : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]), "+v"(acc[4])::"memory");
                CWICK_ROLES_FOLD4("v_mul_f32_dpp", "=v", r0, 0, 1, 2, 3, 0);
                CWICK_ROLES_FOLD4("v_fmac_f32_dpp", "+v", r0, 4, 5, 6, 7, 1);
                CWICK_ROLES_FOLD4("v_fmac_f32_dpp", "+v", r0, 8, 9, 10, 11, 2);
                CWICK_ROLES_FOLD4("v_fmac_f32_dpp", "+v", r0, 12, 13, 14, 15, 3);
                CWICK_ROLES_FOLD4("v_fmac_f32_dpp", "+v", r1, 0, 1, 2, 3, 4);
#undef CWICK_ROLES_FOLD4
#undef CWICK_ROLES_FOLD
#undef CWICK_ROLES_PAIR
                S = (f32x4){sum[0], sum[1], sum[2], sum[3]};
            }
            if constexpr (FLAGS) {
                // did any scoring wave move its reference in tile t?  (rare after the first tiles)
                if (__builtin_amdgcn_readfirstlane(fl[0] | fl[1]) != 0u) {
                    const f32x4 ml = LDS_AT(lds_f32x4, xb + xmr_off);
                    const float m_new = fmaxf(mr, fmaxf(fmaxf(ml[0], ml[1]), fmaxf(ml[2], ml[3])));
                    const float mo = kb == 0 ? ml[0] : kb == 1 ? ml[1] : kb == 2 ? ml[2] : ml[3];
                    const float fo = mo == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mo - m_new);
                    const float c = mr == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(mr - m_new);
                    l_priv = l_priv * c + fo * l_pend;
                    mr = m_new;
                } else {
                    l_priv += l_pend;
                }
            }
            if constexpr (SCORE) {
                // masked positions: past the end of the list (only the last tile of a dense list),
                // or entries of sel[] that name no row
                if (SEL ? true : (!STEADY && ragged && t + 1 == tail_tile)) {
                    uint64_t valid;
                    if (SEL) {
                        const u32x2 vw = LDS_AT(lds_u32x2, tb + VALID_OFF);
                        valid = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)vw[0]) |
                                ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)vw[1]) << 32);
                    } else {
                        valid = __ballot(row_of(t + 1, lane) >= 0);
                    }
                    if (valid != ~0ull) {
                        const uint32_t bits = (uint32_t)(valid >> (16 * kb)) >> (4 * g);
#pragma unroll
                        for (int i = 0; i < 4; i++)
                            if (!((bits >> i) & 1u)) S[i] = -INFINITY;
                    }
                }
                float lmax = vmax3(S[0], S[1], vmax(S[2], S[3])) * c0;    // S stays unscaled: c0 > 0 goes into the exponent's multiply-add
                float m_loc = mr;
                const bool moves = __any(lmax > mr + LAZY);   // rare after the first tiles: only then the lanes of a head confer
                if (moves) {
                    lmax = xor16_max(lmax);
                    lmax = xor32_max(lmax);
                    m_loc = lmax > mr + LAZY ? lmax : mr;
                }
                const float m_use = m_loc == -INFINITY ? 0.0f : m_loc;
                f32x4 P;
#pragma unroll
                for (int i = 0; i < 4; i++) P[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(S[i], c0, -m_use));
                l_pend = (P[0] + P[1]) + (P[2] + P[3]);   // of this lane's four keys, relative to m_loc
                {
                    u32x2 d;
                    d[0] = pack_f16_rne(P[0], P[1]);
                    d[1] = pack_f16_rne(P[2], P[3]);
                    LDS_AT(lds_u32x2, xn + xp_off) = d;
                }
                // the reference this key block used (the four lanes of a head write the same word)
                // and whether it differs from the one every wave holds
                LDS_AT(lds_f32, xn + xm_off) = m_loc;
                LDS_AT(lds_u8, xn + xf_off) = moves ? 1 : 0;
            }
            // the copies this wave issued a step ago (its share of tile t+2) have long landed (in step -1 tile 1 is
            // needed); its share of tile t+3 goes out now, when the wave would otherwise wait at the barrier
            if (!FLAGS && n_tiles > 2) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
            else if (SCORE) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (STEADY) share_steady(t + 3, {r_cp, -1}, lds0 + (uint32_t)((t + 3) & (NST - 1)) * TILE_B);
            else if (do_copy) share(t + 3, {SEL ? r_cp : row_of(t + 3, key_of), -1}, lds0 + (uint32_t)((t + 3) & (NST - 1)) * TILE_B);
            if constexpr (!SCORE) {
                // the sums of the scoring role go where tile t + 1 would have its weights
                float *lsum = reinterpret_cast<float *>(&sm.x[(t + 1) & 1]);      // [head half][head][key block]
                float ls = xor16_sum(l_priv);
                ls = xor32_sum(ls);
                if (g == 0) lsum[(hh * 16 + n) * 4 + kb] = ls;
            }
            LDS_BARRIER();
        };
        int t = 0;
        step(-1, std::integral_constant<int, FIRST>{});
#pragma clang loop unroll(disable)
        for (; t < n_steady; t++) step(t, std::integral_constant<int, STEADY_>{});
#pragma clang loop unroll(disable)
        for (; t + 1 < n_tiles; t++) step(t, std::integral_constant<int, TAIL>{});
        step(t, std::integral_constant<int, LAST>{});
    } else {
        LDS_BARRIER();                                // before copies or weights land in the park area
        f32x4 oacc[2][8];                                 // [head half][dim block]: dims 128 cw + 16 j + 4 g + i, head n
#pragma unroll
        for (int h2 = 0; h2 < 2; h2++)
#pragma unroll
            for (int j = 0; j < 8; j++) oacc[h2][j] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
        int e_run = E_NONE;                               // 2^e_run is above every scale of this wave's block seen so far
        uint32_t thr_bits = 0u;                           // bits of 2^e_run: a scale whose bits reach them does not fit
        float wfac = 0.0f;                                // 2^(WEXP - e_run)
        // the value wave shares its SIMD with two scoring waves that stream MFMAs: without priority
        // its many short VALU instructions wait behind them and it becomes the long pole of the step
        __builtin_amdgcn_s_setprio(3);
        // transpose-read addressing for V^T: lane i of 16-lane group g supplies key 8 g + (i >> 1),
        // bytes 8 (i & 1) .. +7 of the sixteen-byte column
        // (columns 8 cw + j and j + 4 of keys 8 g .. and 32 + 8 g ..: one offset for each j < 4)
        uint32_t tr_off[4];
#pragma unroll
        for (int j = 0; j < 4; j++) tr_off[j] = (uint32_t)(8 * cw + g) * 1024 + place(j, 8 * (g & 1) + (n >> 1), 8) + 8 * (n & 1);
        // the two scales this lane turns into a pair of factors (see the loop)
        const uint32_t sv_off = SC_OFF + (uint32_t)(cw * (TK * 4) + (32 * ((n & 7) >> 2) + 8 * g + 2 * (n & 3)) * 4);
        // the probabilities of this lane's slots: [head half][key half][g][n][4 dwords]
        const uint32_t pw_off = (uint32_t)((g * 16 + n) * 16);
        const uint32_t xml_off = XM_OFF + (uint32_t)(n * 16);
        asm volatile("" ::: "memory");
        // What a tile's values need besides the probabilities is fetched and prepared a step ahead, when the tile is whole
        // already: behind the barrier a step has the probabilities and flags to wait for, and nothing else.  (In step 0
        // that is a round trip to LDS, the first normaliser and eight pairs of factors, 1 200 of the 15 700 cycles of a
        // workgroup with one tile: the value waves have nothing to do while that tile is scored.)
        i32x2 vt[16];                                     // V^T, fragment q: dim block (q >> 1) & 7 of the wave's, key half q & 1
        u32x4 sw[2];                                      // scale * 2^(WEXP - e_run) of the slots' keys, fp16 pairs
        float ecorr = 1.0f;
        auto prepare = [&](int t) {
            const uint32_t tb = lds0 + (uint32_t)(t & (NST - 1)) * TILE_B;
            // The sixteen lanes of a row share their contraction slots (keys 8 g .. 8 g + 7 of each
            // half), so a row needs eight fp16 pairs of scale factors per tile: lane (g, n) reads
            // the two scales of pair n & 7 (half (n & 7) >> 2, keys 8 g + 2 (n & 3) and the next),
            // forms that one pair, and every lane takes the eight pairs out of the row by DPP.
            const f32x2 sv = LDS_AT(lds_f32x2, tb + sv_off);
            const uint32_t va[4] = {tb + tr_off[0], tb + tr_off[1], tb + tr_off[2], tb + tr_off[3]};
#pragma unroll
            for (int q = 0; q < 16; q++) {
                const int j = q >> 1;
                vt[q] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_i32x2 *)(size_t)(va[j & 3] + (uint32_t)(512 * (j >> 2) + 4096 * (q & 1))));
            }
            __builtin_amdgcn_sched_barrier(0);
            // normaliser of the fp16 weights: a power of two above every scale seen so far (it
            // only grows, and only then the lanes confer).  Scales are compared as integers:
            // they are positive, and a negative or NaN scale has the larger bit pattern too.
            ecorr = 1.0f;
            {
                const uint32_t b0 = __builtin_bit_cast(uint32_t, sv[0]) & 0x7FFFFFFFu, b1 = __builtin_bit_cast(uint32_t, sv[1]) & 0x7FFFFFFFu;
                const uint32_t smax = b0 > b1 ? b0 : b1;
                if (__any(smax >= thr_bits && smax != 0u)) {
                    float sm_f = __builtin_bit_cast(float, smax);
                    sm_f = wave_max(sm_f);
                    const int e_tile = (int)((__builtin_bit_cast(uint32_t, sm_f) >> 23) & 0xFFu) - 126;
                    if (e_tile > e_run) {
                        if (e_run != E_NONE) ecorr = pow2i(e_run - e_tile);
                        e_run = e_tile;
                        thr_bits = __builtin_bit_cast(uint32_t, pow2i(e_run));
                        wfac = pow2i(WEXP - e_run);
                    }
                }
            }
            const uint32_t my_pair = pack_f16_rne(sv[0] * wfac, sv[1] * wfac);
            sw[0][0] = row_place<0>(my_pair);
            sw[0][1] = row_place<1>(my_pair);
            sw[0][2] = row_place<2>(my_pair);
            sw[0][3] = row_place<3>(my_pair);
            sw[1][0] = row_place<4>(my_pair);
            sw[1][1] = row_place<5>(my_pair);
            sw[1][2] = row_place<6>(my_pair);
            sw[1][3] = row_place<7>(my_pair);
        };
        // step -1: tile 1 must be whole at the barrier (tile 0 is)
        prepare(0);
        if (n_tiles > 2) CWICK_ROLES_WAIT(0, 2, 3);
        else CWICK_ROLES_WAIT(0, 0, 0);
        RowPair r_cp = {-1, -1};
        if (SEL) r_cp = rows_of(3);                       // rows of the tile copied in step 0; a list entry is a load: fetched a step ahead
        LDS_BARRIER();
        auto step = [&](int t, auto kind) {
            constexpr bool STEADY = decltype(kind)::value == STEADY_;
            const bool do_copy = STEADY || t + 3 < n_tiles;
            {
                // ---- values O^T[dim][head] += V^T W^T for dims 128 cw.., all 32 heads, tile t ----
                const uint32_t xb = lds0 + X_OFF + (uint32_t)(t & 1) * XCH_B;
                const u32x2 fl = LDS_AT(lds_u32x2, xb + XF_OFF);
                u32x4 pw[2][2];                           // [head half][key half]
#pragma unroll
                for (int h2 = 0; h2 < 2; h2++)
#pragma unroll
                    for (int kh = 0; kh < 2; kh++) pw[h2][kh] = LDS_AT(lds_u32x4, xb + pw_off + (uint32_t)((h2 * 2 + kh) * 1024));
                __builtin_amdgcn_sched_barrier(0);
                const uint32_t stage = lds0 + (uint32_t)((t + 3) & (NST - 1)) * TILE_B;   // which tile t-1 left at the last barrier
                if (STEADY) share_steady(t + 3, r_cp, stage);
                else if (do_copy) share(t + 3, SEL ? r_cp : rows_of(t + 3), stage);
                if (SEL && do_copy) r_cp = rows_of(t + 4);
                if (__builtin_amdgcn_readfirstlane(fl[0] | fl[1]) != 0u || ecorr != 1.0f) {
                    // a scoring wave left the common reference in this tile (or the weights'
                    // normaliser grew): bring accumulators and probabilities to the new maximum
#pragma unroll
                    for (int h2 = 0; h2 < 2; h2++) {
                        const f32x4 ml = LDS_AT(lds_f32x4, xb + xml_off + (uint32_t)(h2 * 256));
                        const float m_new = fmaxf(m_ref[h2], fmaxf(fmaxf(ml[0], ml[1]), fmaxf(ml[2], ml[3])));
                        float f[4];
#pragma unroll
                        for (int k = 0; k < 4; k++) f[k] = ml[k] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml[k] - m_new);
                        const float c = (m_ref[h2] == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m_ref[h2] - m_new)) * ecorr;
                        m_ref[h2] = m_new;
                        if (t > 0)
#pragma unroll
                            for (int j = 0; j < 8; j++) oacc[h2][j] *= c;
                        // probabilities were taken relative to each key block's own reference: bring
                        // them to m_new (slot group g of half kh holds keys of key block 2 kh + g / 2)
                        const float fsel0 = (g >> 1) ? f[1] : f[0];
                        const float fsel1 = (g >> 1) ? f[3] : f[2];
#pragma unroll
                        for (int kh = 0; kh < 2; kh++)
#pragma unroll
                            for (int d = 0; d < 4; d++) pw[h2][kh][d] = scale_f16x2(pw[h2][kh][d], kh ? fsel1 : fsel0);
                    }
                }
#pragma unroll
                for (int h2 = 0; h2 < 2; h2++)
#pragma unroll
                    for (int kh = 0; kh < 2; kh++)
#pragma unroll
                        for (int d = 0; d < 4; d++) pw[h2][kh][d] = mul_f16x2(pw[h2][kh][d], sw[kh][d]);
#pragma unroll
                for (int q = 0; q < 16; q++) {
                    const int j = q >> 1, kh = q & 1;
                    u32x4 vh;
                    vh[0] = e4m3x2_to_f16x2<false>((uint32_t)vt[q][0]);
                    vh[1] = e4m3x2_to_f16x2<true>((uint32_t)vt[q][0]);
                    vh[2] = e4m3x2_to_f16x2<false>((uint32_t)vt[q][1]);
                    vh[3] = e4m3x2_to_f16x2<true>((uint32_t)vt[q][1]);
                    const f16x8 v = __builtin_bit_cast(f16x8, vh);
                    oacc[0][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v, __builtin_bit_cast(f16x8, pw[0][kh]), oacc[0][j], 0, 0, 0);
                    oacc[1][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v, __builtin_bit_cast(f16x8, pw[1][kh]), oacc[1][j], 0, 0, 0);
                }
            }
            if (STEADY || t + 1 < n_tiles) prepare(t + 1);
            // tile t+2 must be whole at the next barrier; the share of the tile behind it may stay in flight
            if (do_copy) CWICK_ROLES_WAIT(0, 2, 3);
            else CWICK_ROLES_WAIT(0, 0, 0);
            LDS_BARRIER();
        };
        int t = 0;
#pragma clang loop unroll(disable)
        for (; t < n_steady; t++) step(t, std::integral_constant<int, STEADY_>{});
#pragma clang loop unroll(disable)
        for (; t < n_tiles; t++) step(t, std::integral_constant<int, TAIL>{});

        // ---- every value wave owns its dims: write the partial (or the result) directly ----
        const float *lsum = reinterpret_cast<const float *>(&sm.x[n_tiles & 1]);   // written in front of the last barrier
        const float unit_f = e_run == E_NONE ? 0.0f : pow2i(e_run - WEXP);   // the accumulators are in units of 2^(e_run - WEXP)
        if (n_splits == 1) {
#pragma unroll
            for (int h2 = 0; h2 < 2; h2++) {
                const f32x4 lv = *(const f32x4 *)&lsum[(h2 * 16 + n) * 4];
                float L = (lv[0] + lv[1]) + (lv[2] + lv[3]);
                const int head = hb * HW + 16 * h2 + n;
                if (head >= nh) continue;
                // the attention sink of src/ds_model.c:946: one more term in the denominator, no value
                // (with several splits the merge kernel adds it)
                if (p.sink && m_ref[h2] > -INFINITY)
                    L += __builtin_amdgcn_exp2f(p.sink[head] * 1.44269504088896340736f - m_ref[h2]);
                const float fin = L > 0.0f ? unit_f / L : 0.0f;
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    // accumulator register i <-> dim 16 db + 4 g + i
                    const f32x4 v = oacc[h2][j] * fin;
                    *(f32x4 *)(p.out + (size_t)(y * (uint32_t)nh + (uint32_t)head) * VDIM + 16 * (8 * cw + j) + 4 * g) = v;
                }
            }
            return;
        }
        // The partial leaves as 16-bit fixed point: this wave's 128 dims of the head share one scale, their largest
        // magnitude, so every value is off by at most 2^-16 of that.  A non-finite value makes the scale NaN and with it
        // the head's merged output (v_maximum3 hands a NaN on; two values and their signs an instruction, four
        // chains, because each link waits for the one before it; the four lanes of a head meet without a trip through
        // LDS).
        float big[2];
        const size_t pb0 = (size_t)(y * (uint32_t)n_splits + (uint32_t)split) * (2 * n_hb) + 2 * hb;
#pragma unroll
        for (int h2 = 0; h2 < 2; h2++) {
            float m[4];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const f32x4 a = oacc[h2][2 * c], b = oacc[h2][2 * c + 1];
                m[c] = maximum3_abs(a[0], a[1], a[2]);
                m[c] = maximum3_abs(m[c], a[3], b[0]);
                m[c] = maximum3_abs(m[c], b[1], b[2]);
                m[c] = maximum3_abs(m[c], b[3], b[3]);
            }
            uint32_t bm = __builtin_bit_cast(uint32_t, maximum3_abs(maximum3_abs(m[0], m[1], m[2]), m[3], m[3])) & 0x7FFFFFFFu;
            bm = lanes_xor16_max(bm);                     // (as integers: NaNs and infinities are above every finite value)
            bm = lanes_xor32_max(bm);
            big[h2] = bm > 0x7F7FFFFFu ? __builtin_nanf("") : __builtin_bit_cast(float, bm);   // in accumulator units
            const float to_unit = big[h2] > 0.0f ? 1.0f / big[h2] : 0.0f;
            if (hb * HW + 16 * h2 + n < nh) {
                uint32_t *pq = p.part_acc + ((pb0 + h2) * NDB + 8 * cw) * 128 + lane * 2;   // [db][lane][4 x i16]
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const f32x4 v = oacc[h2][j] * to_unit;
                    u32x2 w;
                    w[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pknorm_i16(v[0], v[1]));
                    w[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pknorm_i16(v[2], v[3]));
                    store_through8(pq + j * 128, w);
                }
            }
        }
        if (g < 2 && hb * HW + 16 * g + n < nh) {
            const f32x4 lv = *(const f32x4 *)&lsum[lane * 4];
            const float L = (lv[0] + lv[1]) + (lv[2] + lv[3]);
            *(f32x4 *)(p.part_ml + (((pb0 + (uint32_t)g) * 4 + cw) * HB + n) * 4) =
                (f32x4){(g ? m_ref[1] : m_ref[0]) * 0.69314718055994530942f, L, (g ? big[1] : big[0]) * unit_f * (1.0f / 32767.0f), 0.0f};
        }
    }
}

// merge of fragment-layout partials: values [y][split][16-head block][dim block][lane][4], as 16-bit
// fixed point (the decode's) or fp32 (the chunk prefill's), and per 16-head block and quarter of the
// dims [head][4] floats (running maximum in natural-log units, weight sum, value of one fixed-point step
// or unit of the accumulators, unused).  With more
// than eight splits a workgroup is one dim block of one 16-head block: its waves (eight up to
// 64 splits, where a wave then has its eight loads in flight at once: 4.55 -> 4.16 us; sixteen
// beyond) take splits w, w + n_waves, ... and meet in LDS.  With up to eight a wave merges a dim block alone and
// eight of them make a workgroup (a batch of queries splits each query less: one wave per
// split would be thousands of workgroups that each wait out one load).  Every wave has all its
// loads in flight at once (eight splits per batch); which splits exist is uniform per wave, so
// absent ones cost nothing.
constexpr int MW = 16;
// (the kernel goes by these too: an argument behind the first fourteen dwords, or the launch's own sizes, would be a
// trip to memory in front of the first load)
__host__ __device__ inline bool merge_packed(int n_splits) { return n_splits <= 8; }
__host__ __device__ inline int merge_waves(int n_splits) { return n_splits <= 64 ? 8 : MW; }
__device__ __forceinline__ f32x4 part_value(const u32x2 a) {
    return (f32x4){(float)((int32_t)(a[0] << 16) >> 16), (float)((int32_t)a[0] >> 16),
                   (float)((int32_t)(a[1] << 16) >> 16), (float)((int32_t)a[1] >> 16)};
}
__device__ __forceinline__ f32x4 part_value(const f32x4 a) { return a; }
// what each row of sixteen lanes holds, in all of them
__device__ __forceinline__ void rows_to_all(float x, float (&out)[4]) {
    uint32_t a = __builtin_bit_cast(uint32_t, x), b = a;
    lanes_swap32(a, b);                                 // a: rows 0, 1, 0, 1; b: rows 2, 3, 2, 3
    uint32_t c = a, d = b;
    lanes_swap16(a, c);
    lanes_swap16(b, d);
    out[0] = __builtin_bit_cast(float, a), out[1] = __builtin_bit_cast(float, c);
    out[2] = __builtin_bit_cast(float, b), out[3] = __builtin_bit_cast(float, d);
}
template <class PART>                             // u32x2: four 16-bit values; f32x4
__device__ __forceinline__ void
merge_frag(const PART *__restrict__ part_acc, const float *__restrict__ part_ml, int n_splits, int n_hb16, int nhb,
           uint32_t n_rb, int nh, const float *__restrict__ sink, float *__restrict__ out) {
    __shared__ float red_m[MW][64];
    __shared__ float red_l[MW][64];
    __shared__ f32x4 red_a[MW][64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), y = blockIdx.y;
    int wv, mw, db, hb;
    if (merge_packed(n_splits)) {
        // up to eight splits: a wave merges a dim block by itself, and the workgroup's eight
        // waves take the eight dim blocks of one quarter
        wv = 0, mw = 1, db = 8 * (int)(blockIdx.x & 3) + wave, hb = (int)(blockIdx.x >> 2);
    } else {
        // workgroups go to the eight XCDs round robin: the eight dim blocks that share a quarter's
        // [head][4] floats sit on one XCD, so that only one L2 fetches them (with an odd number of
        // row blocks on two)
        const int b = (int)blockIdx.x, grp = n_hb16 & 1 ? (b & 3) + 4 * (b >> 5) : (b & 7) + 8 * (b >> 6);
        wv = wave, mw = merge_waves(n_splits);
        db = 8 * (grp & 3) + ((n_hb16 & 1 ? b >> 2 : b >> 3) & 7), hb = grp >> 2;
    }
    const int n = lane & 15, g = lane >> 4;
    const size_t sb = (size_t)y * n_splits;
    const float *ml = part_ml + (((sb * n_hb16 + hb) * 4 + (db >> 3)) * HB + n) * 4;
    const size_t ml_stride = (size_t)n_hb16 * 4 * HB * 4;
    const PART *pa = part_acc + ((sb * n_hb16 + hb) * NDB + db) * 64 + lane;
    const size_t pa_stride = (size_t)n_hb16 * NDB * 64;

    // Four slices come with one load of [head][4] floats, a row of sixteen lanes for each (a load of the same
    // sixteen heads for all four rows takes the memory pipeline as long), and what the values are weighted by goes to
    // the other rows by swaps.  48 slices of 64 heads: 4.0 us with a load for each slice, 3.5 so.
    PART a0[8];
    f32x4 v0[2];
    auto fetch = [&](int s0, auto count) {
#pragma unroll
        for (int i = 0; i < decltype(count)::value / 4; i++) {
            const int s = s0 + mw * (4 * i + g);
            v0[i] = *(const f32x4 *)(ml + (s < n_splits ? s : n_splits - 1) * ml_stride);
        }
#pragma unroll
        for (int j = 0; j < decltype(count)::value; j++) {
            const int s = s0 + mw * j;
            a0[j] = pa[(s < n_splits ? s : n_splits - 1) * pa_stride];
        }
#pragma unroll
        for (int i = 0; i < decltype(count)::value / 4; i++)
            if (s0 + mw * (4 * i + g) >= n_splits) v0[i] = (f32x4){-INFINITY, 0.0f, 0.0f, 0.0f};
    };
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    float ls = 0.f, mx = -INFINITY;                   // ls: of this row's slices
    auto add = [&](auto count) {
#pragma unroll
        for (int i = 0; i < decltype(count)::value / 4; i++) {
            const float c = v0[i][0] == -INFINITY ? 0.0f : __expf(v0[i][0] - mx);
            ls = __builtin_fmaf(v0[i][1], c, ls);
            float cs[4];
            rows_to_all(c * v0[i][2], cs);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const f32x4 x = part_value(a0[4 * i + j]);
#pragma unroll
                for (int r = 0; r < 4; r++) acc[r] = __builtin_fmaf(x[r], cs[j], acc[r]);
            }
        }
    };
    auto meet = [&] {
        mx = xor32_max(xor16_max(mx));
        if (mw > 1) {
            red_m[wv][lane] = mx;
            __syncthreads();
            for (int w = 0; w < mw; w++) mx = fmaxf(mx, red_m[w][lane]);
        }
    };
    const std::integral_constant<int, 4> four;
    const std::integral_constant<int, 8> eight;
    if (n_splits <= 4 * mw) {
        fetch(wv, four);
        mx = v0[0][0];
        meet();
        add(four);
    } else {
        fetch(wv, eight);
        mx = fmaxf(v0[0][0], v0[1][0]);
        for (int s = wv + mw * (8 + g); s < n_splits; s += 4 * mw) mx = fmaxf(mx, ml[s * ml_stride]);
        meet();
        add(eight);
        for (int s0 = wv + 8 * mw; s0 < n_splits; s0 += 8 * mw) {
            fetch(s0, eight);
            add(eight);
        }
    }
    ls = xor32_sum(xor16_sum(ls));
    float l = ls;
    f32x4 r4 = acc;
    if (mw > 1) {
        red_l[wv][lane] = ls;
        red_a[wv][lane] = acc;
        __syncthreads();
        if (wv != 0) return;
        l = 0.f;
        r4 = (f32x4){0.f, 0.f, 0.f, 0.f};
        for (int w = 0; w < mw; w++) {
            l += red_l[w][lane];
            const f32x4 t = red_a[w][lane];
#pragma unroll
            for (int r = 0; r < 4; r++) r4[r] += t[r];
        }
    }
    // row block hb of group y: heads 16 (rb % nhb) .. of query rb / nhb
    const uint32_t rb = (uint32_t)y * (uint32_t)n_hb16 + (uint32_t)hb, yq = rb / (uint32_t)nhb;
    const int head = (int)(rb - yq * (uint32_t)nhb) * HB + n;
    if (rb >= n_rb || head >= nh) return;
    if (sink && mx > -INFINITY) l += __expf(sink[head] - mx);
    const float inv = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
    for (int r = 0; r < 4; r++) r4[r] *= inv;
    // accumulator register i <-> dim 16 db + 4 g + i
    *(f32x4 *)(out + ((size_t)yq * nh + head) * VDIM + 16 * db + 4 * g) = r4;
}
__global__ void __launch_bounds__(64 * MW)
mla_merge_frag16_kernel(const u32x2 *__restrict__ part_acc, const float *__restrict__ part_ml, int n_splits, int n_hb16,
                        int nhb, uint32_t n_rb, int nh, const float *__restrict__ sink, float *__restrict__ out) {
    merge_frag(part_acc, part_ml, n_splits, n_hb16, nhb, n_rb, nh, sink, out);
}
__global__ void __launch_bounds__(64 * MW)
mla_merge_frag32_kernel(const f32x4 *__restrict__ part_acc, const float *__restrict__ part_ml, int n_splits, int n_hb16,
                        int nhb, uint32_t n_rb, int nh, const float *__restrict__ sink, float *__restrict__ out) {
    merge_frag(part_acc, part_ml, n_splits, n_hb16, nhb, n_rb, nh, sink, out);
}

// Split-K partials of the entry point that may not allocate (cwick_hip_mla_decode_static_dev):
// a fixed area in the library's own device image instead of the grow-only workspace.  Host code
// never uses the array's name as an address: static_scratch() asks the runtime once where the
// device's copy lives and hands out that pointer.
constexpr size_t STATIC_SCRATCH_BYTES = (size_t)16 << 20;
static __device__ __align__(256) unsigned char scratch[STATIC_SCRATCH_BYTES];

static void *static_scratch() {
    static std::once_flag once;
    static void *ptr = nullptr;
    static hipError_t err = hipSuccess;
    std::call_once(once, [] {
        err = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (err != hipSuccess) ptr = nullptr;
    });
    if (!ptr) hip_ok(err != hipSuccess ? err : hipErrorInvalidSymbol, "hipGetSymbolAddress(scratch)");
    return ptr;
}

}  // namespace

template <class PART>
static int launch_merge_of(void (*kernel)(const PART *, const float *, int, int, int, uint32_t, int, const float *, float *),
                           const PART *part_acc, const float *part_ml, int n_splits, int n_groups, int n_hb16, int nhb,
                           int64_t n_rb, int nh, const float *sink, float *out, int prof, hipStream_t s) {
    ProfKernel pk(prof, s);
    pk.launch(kernel, dim3(n_hb16 * (merge_packed(n_splits) ? 4 : NDB), n_groups), dim3(64 * merge_waves(n_splits)), 0,
              part_acc, part_ml, n_splits, n_hb16, nhb, (uint32_t)n_rb, nh, sink, out);
    CWICK_HIP_CALL(hipGetLastError());
    return 1;
}
int launch_mla_merge(const u32x2 *part_acc, const float *part_ml, int n_splits, int n_groups, int n_hb16, int nhb,
                     int64_t n_rb, int nh, const float *sink, float *out, int prof, hipStream_t s) {
    return launch_merge_of(mla_merge_frag16_kernel, part_acc, part_ml, n_splits, n_groups, n_hb16, nhb, n_rb, nh, sink, out, prof, s);
}
int launch_mla_merge(const f32x4 *part_acc, const float *part_ml, int n_splits, int n_groups, int n_hb16, int nhb,
                     int64_t n_rb, int nh, const float *sink, float *out, int prof, hipStream_t s) {
    return launch_merge_of(mla_merge_frag32_kernel, part_acc, part_ml, n_splits, n_groups, n_hb16, nhb, n_rb, nh, sink, out, prof, s);
}

namespace {

// fixed == true: partials go to the static area, nothing is allocated and no events are created
int run(Params &p, int most_splits, hipStream_t s, bool fixed) {
    static std::once_flag attr_once;
    static hipError_t attr_err = hipSuccess;
    const size_t smem = sizeof(Smem);
    std::call_once(attr_once, [&] {
        attr_err = hipFuncSetAttribute((const void *)mla_roles_kernel<false>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
        if (attr_err == hipSuccess)
            attr_err = hipFuncSetAttribute((const void *)mla_roles_kernel<true>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    });
    CWICK_HIP_CALL(attr_err);
    const int n_hb = (p.nh + HW - 1) / HW;
    const int64_t total = (int64_t)n_hb * p.n_splits * p.nq;     // below 2^25: n_hb <= 4, and splits only up to the compute units
    CWICK_REQUIRE(total < (1 << 25), "mla: grid of %lld workgroups is too large", (long long)total);
    if (p.n_splits > 1) {
        const size_t acc_b = (size_t)p.nq * p.n_splits * n_hb * HW * VDIM * sizeof(int16_t);
        const size_t ml_b = (size_t)p.nq * p.n_splits * n_hb * HW * 4 * 4 * sizeof(float);
        char *ws;
        if (fixed) {
            CWICK_REQUIRE(acc_b + ml_b <= STATIC_SCRATCH_BYTES,
                          "mla_decode_static: the split-K partials of this call (%zu bytes) exceed the "
                          "static scratch area (%zu bytes); use cwick_hip_mla_decode_dev",
                          acc_b + ml_b, STATIC_SCRATCH_BYTES);
            ws = (char *)static_scratch();
            if (!ws) return 0;
        } else {
            // (asked for: as many splits as any call of up to this many keys has)
            ws = (char *)workspace(s, (acc_b + ml_b) / p.n_splits * most_splits);
            if (!ws) return 0;                      // workspace() has recorded why
        }
        p.rest.part_acc = (uint32_t *)ws;
        p.rest.part_ml = (float *)(ws + acc_b);
    }
    {
        ProfKernel pk(fixed ? -1 : CWICK_HIP_PROF_MLA, s);
        pk.launch(p.sel ? mla_roles_kernel<true> : mla_roles_kernel<false>, dim3((unsigned)total), dim3(THREADS), smem,
                  p.q, p.rows, p.scales, p.sel, (uint32_t)p.n_list, (uint32_t)p.n_rows, (uint32_t)p.keys_per_split,
                  (uint32_t)p.nh | (uint32_t)p.n_splits << 8, div_inverse((uint32_t)p.n_splits),
                  total % 8 == 0 ? (uint32_t)(total / 8) : 0u, p.rest);
    }
    CWICK_HIP_CALL(hipGetLastError());
    if (p.n_splits > 1)
        return launch_mla_merge((const u32x2 *)p.rest.part_acc, p.rest.part_ml, p.n_splits, p.nq, 2 * n_hb, 2 * n_hb, (int64_t)p.nq * 2 * n_hb, p.nh,
                                p.rest.sink, p.rest.out, fixed ? -1 : CWICK_HIP_PROF_MLA_MERGE, s);
    return 1;
}

int splits_per_cu() {
    static const int v = [] {
        const char *e = getenv("CWICK_HIP_MLA_WG_PER_CU");
        const int x = e ? atoi(e) : 1;
        return (x < 1 || x > 8) ? 1 : x;
    }();
    return v;
}

}  // namespace

int launch_mla_decode(const uint8_t *rows, const float *scales, int64_t row_bstride,
                      int64_t scale_bstride, int64_t n_rows, int batch, const int32_t *sel,
                      int64_t n_list, const uint16_t *q, int n_heads, float scale, const float *sink,
                      float *out, hipStream_t s, bool fixed_scratch) {
    CWICK_REQUIRE(rows && scales && q && out, "mla_decode: null pointer");
    CWICK_REQUIRE(batch >= 1 && batch <= 4096, "mla_decode: batch %d", batch);
    CWICK_REQUIRE(n_heads >= 1 && n_heads <= 128, "mla_decode: n_heads %d (1..128)", n_heads);
    CWICK_REQUIRE(n_rows >= 1 && n_rows <= ((int64_t)1 << 31) - 1, "mla_decode: n_rows %lld",
                  (long long)n_rows);
    CWICK_REQUIRE(n_list >= 1 && n_list <= ((int64_t)1 << 31) - 1, "mla_decode: n_list %lld",
                  (long long)n_list);
    CWICK_REQUIRE(sel || n_list <= n_rows, "mla_decode: n_list %lld exceeds n_rows %lld",
                  (long long)n_list, (long long)n_rows);
    CWICK_REQUIRE(scale > 0.0f && scale < INFINITY, "mla_decode: scale must be positive");
    CWICK_REQUIRE((uintptr_t)rows % 16 == 0 && row_bstride % 16 == 0 && (uintptr_t)q % 16 == 0 &&
                      (uintptr_t)out % 16 == 0 && (uintptr_t)scales % 4 == 0,
                  "mla_decode: rows, q and out must be 16-byte aligned");
    Params p{};
    p.rows = rows; p.scales = scales; p.n_rows = n_rows; p.sel = sel; p.n_list = n_list;
    p.q = q; p.nh = n_heads; p.nq = batch;
    p.rest.row_bstride = row_bstride; p.rest.scale_bstride = scale_bstride;
    p.rest.scale = scale; p.rest.out = out; p.rest.sink = sink;
    const int n_hb = (n_heads + HW - 1) / HW;
    const int64_t tiles = (n_list + TK - 1) / TK, want = mla_decode_most_splits(n_hb * batch, splits_per_cu(), num_cus());
    const int64_t per = (int64_t)TK * mla_decode_tiles(tiles, n_hb * batch, sel != nullptr, splits_per_cu(), num_cus());
    p.keys_per_split = per;
    p.n_splits = (int)((n_list + per - 1) / per);
    return run(p, (int)(tiles < want ? tiles : want), s, fixed_scratch);
}

}  // namespace cwick
