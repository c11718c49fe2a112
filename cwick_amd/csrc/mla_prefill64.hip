// mla_prefill64.hip -- absorbed-latent MLA chunked prefill (src/attention.c:1010-1019: one
// mla_latent_decode per query of the chunk, :749-811) with 64 query rows per key tile.
//
// The decode kernel (mla_roles.hip) gives a workgroup 32 heads of one query, and what a 64-key
// tile costs it besides the matrix work -- the copy into LDS, the handling of the block scales,
// the E4M3 -> fp16 conversion of V -- does not depend on the number of rows.  A prefill chunk has
// rows to spare, so here a workgroup takes 64 rows and pays that per twice the matrix work.
//
//   rows come in blocks of sixteen heads of one query, numbered through the chunk; a workgroup
//   takes four consecutive ones (a group): 64 heads of one query, or, with fewer heads, up to four
//   queries that share the tiles and differ in at most three keys (SPAN).  512 queries of 16 heads
//   over 5.5K rows: 227 us with one query per workgroup, 101 so.  Where the groups do not fill the
//   chip a group's keys are cut into slices (mla_plan.hpp) whose fp32 partials mla_merge_frag32_kernel
//   combines: 8 queries of 128 heads over 20K rows 453 -> 55 us, 52 over 13.5K 313 -> 170.
//
//   workgroup = 8 waves (two per SIMD, 256 registers each), 64 rows x all keys of the group,
//   walked in tiles of 64 keys, three LDS stages.
//     waves 0..3 score: wave hq owns row block hq and scores it against all 64 keys of
//                the tile (four 16-key blocks): S^T = K Q^T on v_mfma_scale_f32_16x16x128_f8f6f4,
//                K as stored, Q as two E4M3 terms with one E8M0 scale per head and 128-dim block
//                (as in mla_roles.hip).  The keys' block scales sit in five registers per tile (a
//                key per lane) and enter the fold of the five block products through a DPP row
//                broadcast inside the multiply-add.  Because a wave sees every key of its heads,
//                the softmax reference of a head lives in one wave: when a tile exceeds it by
//                2^LAZY the wave moves it at once, and publishes the factor by which the
//                accumulators of that head shrink together with the fp16 probabilities of the tile.
//     waves 4..7 accumulate: wave cw owns output dims 128 cw .. +127 for all 64 rows;
//                weights p * scale[key][cw] * 2^(10 - e) in fp16, O^T += V^T W^T on
//                v_mfma_f32_16x16x32_f16, every converted V^T fragment used four times.
//   The roles run one tile apart (tile t+1 is scored while tile t is accumulated): one barrier
//   per step.  Tile t+2 is copied (global_load_lds, issued from assembly) at the top of step t
//   into the stage tile t-1 left at the last barrier, by the value waves alone: a wave stalls
//   while the memory pipeline takes its copies, and the scoring waves are the longer pole of a
//   step (copies dealt to all eight waves: 36.1 ms for 4096 queries over 28672 + 4096 rows,
//   by the value waves: 31.2; spreading them over the step or issuing them a step earlier into
//   the columns a value wave has just finished with: 31.1 and 34).
//   A group that is not cut has no partials: the value waves write the output.
//   Per tile the workgroup reads about 275 KB from LDS (160 KB of K fragments, 32 KB of V^T, 32 KB
//   of probabilities, the scale registers) and the copies write 37 KB; with the scales as twenty
//   16-byte fragments per scoring wave it was 350 KB and the kernel 7 % slower.
//   Ablation builds at 31 ms: without the value MFMAs and conversions 21.7, without the score
//   MFMAs and K reads 22.4, without the K reads alone 27.3: the two roles weigh the same and
//   mostly add up; the matrix pipe is busy 2 176 of about 4 200 cycles per step and SIMD.
//   Every K fragment is read from LDS by all four scoring waves (160 KB per tile); a timing build
//   that read half of them ran 11 % faster (3 % since the scales are registers).
#include "common.hpp"
#include "mla_plan.hpp"

#include <mutex>

namespace cwick {
namespace {

constexpr int KDIM = CWICK_HIP_LATENT_KDIM;   // 576
constexpr int VDIM = CWICK_HIP_LATENT_VDIM;   // 512
constexpr int NBLK = CWICK_HIP_LATENT_NBLK;   // 5
constexpr int THREADS = 512;                  // waves 0..3 score, waves 4..7 accumulate values
constexpr int NWAVES = THREADS / 64;
constexpr int TK = 64;                        // keys per tile
constexpr int HW = 64;                        // heads per workgroup
constexpr int NHQ = HW / 16;                  // 16-head blocks = scoring waves
constexpr int NST = 3;                        // tile stages
constexpr int NCOL = KDIM / 16;               // 36 sixteen-byte columns per row
constexpr float LAZY = 10.0f;                 // the reference moves when a tile exceeds it by 2^LAZY (fp16 probabilities up to 2^10)
constexpr int WEXP = 4;                       // fp16 weights are p * scale * 2^(WEXP - e), scale < 2^e: below 2^(LAZY + WEXP) = 2^14
constexpr int E_NONE = -1000;                 // no scale seen yet

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
typedef __attribute__((ext_vector_type(8))) int i32x8;
typedef __attribute__((ext_vector_type(2))) int i32x2;
typedef __attribute__((address_space(3))) i32x2 lds_i32x2;
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) u32x2 lds_u32x2;
typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
typedef __attribute__((address_space(3))) f32x2 lds_f32x2;
typedef __attribute__((address_space(3))) float lds_f32;
typedef __attribute__((address_space(3))) uint32_t lds_u32;

// What a workgroup needs late; the rest are arguments of the kernel's own, in registers (see mla_roles.hip).
struct WideRest {
    float *out;               // [nq][nh][512]
    float *part_ml;           // as in mla_roles.hip, [group of n_rest][slice][row block of the group]
    float *part_acc;
    float scale;
};

// what a position past the end of a query's keys is fetched from (see mla_roles.hip)
__device__ __attribute__((aligned(16))) uint8_t g_zero_row64[KDIM + 64] = {0};
__device__ __attribute__((aligned(16))) float g_zero_scales64[8] = {0.0f};

struct Tile {
    uint8_t kv[NCOL][TK][16];     // [16-byte column][key][16]     36864 B
    float sc[NBLK][TK];           // [block][key]                   1280 B
    uint32_t pad[4];
};
struct Xch {                       // what the scoring waves publish per tile
    // fp16 probabilities exp2(s - m) as the B fragments of the value MFMA:
    // [16-head block][32-key half][slot group g][head n][4 dwords]; contraction slot 8 g + j of a
    // half is key 8 g + j of that half
    uint32_t p[NHQ][2][4][16][4];
    float c[NHQ][16];             // by what the accumulators of head (hq, n) shrink before this tile
    uint32_t moved[NHQ];          // scoring wave hq moved a reference in this tile
    uint32_t pad[12];
};
struct Smem {
    Tile tile[NST];
    Xch x[2];
};
// Q of one (16-head block, 128-dim block), unit u = 5 hq + b: 64 bytes per lane, first as copied from
// memory ([4][lane][16]: the lane's 32 bf16 values), then in MFMA operand order (two sixteen-byte pieces
// of the hi term, two of the lo term; the rope block's one register set in place of its hi term).
// Parked behind the first two tile stages, the scale bytes behind it.
constexpr uint32_t PARK = 2 * (uint32_t)sizeof(Tile), PARK_UNIT = 4096, PARK_LO = 2048;
constexpr uint32_t PARK_SC = PARK + 5 * NHQ * PARK_UNIT, PARK_END = PARK_SC + 5 * NHQ * 256;
constexpr size_t SMEM_BYTES = sizeof(Smem) > PARK_END ? sizeof(Smem) : PARK_END;
static_assert(SMEM_BYTES <= 160 * 1024, "LDS");

__device__ __forceinline__ float pow2i(int e) {
    e = e > 126 ? 126 : (e < -126 ? -126 : e);
    return __builtin_bit_cast(float, (uint32_t)(e + 127) << 23);
}
__device__ __forceinline__ uint32_t mul_f16x2(uint32_t a, uint32_t b) {
    const f16x2 r = __builtin_bit_cast(f16x2, a) * __builtin_bit_cast(f16x2, b);
    return __builtin_bit_cast(uint32_t, r);
}
#define LDS_BARRIER() asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory")
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
#define LDS_AT(type, a) (*(type *)(size_t)(uint32_t)(a))

constexpr uint32_t TILE_B = sizeof(Tile);
constexpr uint32_t SC_OFF = NCOL * TK * 16;                       // Tile::sc
constexpr uint32_t X_OFF = NST * TILE_B;                          // Smem::x
constexpr uint32_t XCH_B = sizeof(Xch);
constexpr uint32_t XC_OFF = NHQ * 2 * 4 * 16 * 4 * 4;             // Xch::c
constexpr uint32_t XF_OFF = XC_OFF + NHQ * 16 * 4;                // Xch::moved

// d = x * r[place n of the row]  /  d += x * r[place n of the row]: the factor comes out of one
// lane of each row of sixteen (DPP row broadcast inside the multiply), so a row's sixteen factors
// live in one register.  Assembly: the compiler folds a DPP move into a multiply but not into a
// multiply-add.  It does not space an assembly statement from an MFMA whose result the statement
// reads: x must have been written at least eleven instructions earlier (an 8-pass MFMA), which
// the callers arrange by the order of their (volatile) statements.
__device__ __forceinline__ void scaled_by_row_lane(float &d, float r, float x, int nsel, bool first) {
#define CWICK_SBL_CASE(n)                                                                                         \
    case n:                                                                                                       \
        if (first) asm volatile("v_mul_f32_dpp %0, %1, %2 row_newbcast:" #n " row_mask:0xf bank_mask:0xf" : "=v"(d) : "v"(r), "v"(x)); \
        else asm volatile("v_fmac_f32_dpp %0, %1, %2 row_newbcast:" #n " row_mask:0xf bank_mask:0xf" : "+v"(d) : "v"(r), "v"(x));      \
        break;
    switch (nsel) {
        CWICK_SBL_CASE(0) CWICK_SBL_CASE(1) CWICK_SBL_CASE(2) CWICK_SBL_CASE(3) CWICK_SBL_CASE(4) CWICK_SBL_CASE(5)
        CWICK_SBL_CASE(6) CWICK_SBL_CASE(7) CWICK_SBL_CASE(8) CWICK_SBL_CASE(9) CWICK_SBL_CASE(10) CWICK_SBL_CASE(11)
        CWICK_SBL_CASE(12) CWICK_SBL_CASE(13) CWICK_SBL_CASE(14) CWICK_SBL_CASE(15)
        default: break;
    }
#undef CWICK_SBL_CASE
}

// The parts that run once per workgroup -- addresses, Q, the output -- are written for few bytes of
// code.  A compute unit starts a launch with a cold instruction cache, and straight-line code costs it
// about 150 cycles per 64 bytes: unrolled, what lies around the loops took 20 000 cycles of a
// workgroup whose key tile takes 4 000.
// q: [nq][nh][576] bf16; query y sees rows 0 .. pos0 + y.  shape: the heads nh of a query in the low eight bits,
// above them the row blocks of a group, gsz: four, or fewer where groups of four leave the chip idle.
// nhb_inv: 2^31 / nhb, rounded up, for the nhb = 16-head blocks of a query.  n_rb: row blocks of the chunk, block rb
// is heads 16 (rb % nhb) .. of query rb / nhb.  The last n_whole groups take a workgroup each; the first n_rest
// take p_slices workgroups each and leave partials; slices_inv as nhb_inv.
template <bool SPAN>
__global__ void __launch_bounds__(THREADS)
mla_prefill64_kernel(const uint16_t *__restrict__ q, const uint8_t *__restrict__ all_rows, const float *__restrict__ all_scales,
                     int pos0, uint32_t shape, uint32_t nhb_inv, uint32_t n_rb, uint32_t n_whole, uint32_t n_rest,
                     uint32_t p_slices, uint32_t slices_inv, const WideRest p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    Smem &sm = *reinterpret_cast<Smem *>(smem_raw);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void *)smem_raw;

    const int nh = (int)(shape & 255u);
    const uint32_t gsz = shape >> 8, nhb = (uint32_t)(nh + 15) / 16;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool scorer = wave < NHQ;
    const int hq = wave & 3;         // scoring role: heads 16 hq .. 16 hq + 15
    const int cw = wave & 3;         // value role: dims 128 cw .. +127 = scale block cw
    const int n = lane & 15;         // head column / key row of a 16-block / dim row
    const int g = lane >> 4;         // 32-wide contraction block (QK) / 8-wide (PV)

    // Workgroups go to the eight XCDs round robin.  The groups of a query run on one XCD (they
    // read the same tiles at the same time: one fetch into that L2), and consecutive queries go
    // to consecutive XCDs, so that every XCD gets the same mix of long and short queries (a
    // contiguous eighth of the queries per XCD left the XCD with the longest ones 6 % behind).
    // The queries with the most keys start first, the groups in slices last.
    uint32_t grp, slice = 0, n_slices = 1;
    const bool sliced = blockIdx.x >= n_whole;
    if (!sliced) {
        uint32_t i = blockIdx.x;
        const uint32_t lg = nhb == 2 * gsz ? 4 : 3, lot = i >> lg, r = i & ((1u << lg) - 1);     // eight queries of one or two groups
        if (((lot + 1) << lg) <= n_whole) i = ((8 * lot + r % 8) << (lg - 3)) + r / 8;
        grp = n_rest + n_whole - 1 - i;
    } else {
        n_slices = p_slices;
        const uint32_t i = blockIdx.x - n_whole, above = div_by(i, slices_inv);
        grp = n_rest - 1 - above;
        slice = i - above * n_slices;
    }
    // the query of row block h of the group (past the end of the chunk: its last row block again, not stored)
    // (and past the end of a smaller group its last one)
    auto rb_of = [&](uint32_t h) -> uint32_t {
        const uint32_t rb = gsz * grp + (h < gsz ? h : gsz - 1);
        return rb < n_rb ? rb : n_rb - 1;
    };
    const int keys_hi = pos0 + 1 + (int)div_by(rb_of(NHQ - 1), nhb_inv);      // of the group's last query
    const uint32_t all_tiles = ((uint32_t)keys_hi + TK - 1) / TK;
    uint32_t t_first = 0, t_end = all_tiles;
    if (sliced) {
        const uint32_t per = div_by(all_tiles + n_slices - 1, slices_inv);
        t_first = slice * per < all_tiles ? slice * per : all_tiles;
        t_end = t_first + per < all_tiles ? t_first + per : all_tiles;
    }
    const int n_tiles = (int)(t_end - t_first);
    // from here on positions count from the slice's first key
    const int key0 = (int)t_first * TK;
    const int n_keys = t_end == all_tiles ? keys_hi - key0 : n_tiles * TK;
    auto keys_of = [&](uint32_t h) -> int { return pos0 + 1 + (int)div_by(rb_of(h), nhb_inv) - key0; };
    const uint8_t *rows = all_rows + (size_t)key0 * KDIM;
    const float *scales = all_scales + (size_t)key0 * NBLK;

    uint64_t zrow = (uint64_t)(uintptr_t)g_zero_row64, zsc = (uint64_t)(uintptr_t)g_zero_scales64;
    asm volatile("" : "+s"(zrow), "+s"(zsc));

    // ---- tile copies.  lane = key of the tile; the 36 sixteen-byte columns and 5 scale blocks are
    // dealt round robin: wave w copies columns w, w + 8, w + 16, w + 24, and w + 32 when w < 4;
    // waves 4..7 scale block w - 4, wave 0 scale block 4.  M0 is written by the statement that
    // needs it (the compiler has no other use of M0 in this file; tests check the compiled code).
    auto dma16 = [&](uint64_t gp, uint32_t lds_off) {
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(gp), "s"(lds_off) : "memory");
    };
    auto dma4 = [&](uint64_t gp, uint32_t lds_off) {
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(gp), "s"(lds_off) : "memory");
    };
    auto share = [&](int t, uint32_t tile_off) {
        const int r = t * TK + lane;
        const bool live = r < n_keys;
        const uint64_t rp = live ? (uint64_t)(uintptr_t)rows + (uint64_t)(uint32_t)r * KDIM : zrow;
        const uint64_t sp = live ? (uint64_t)(uintptr_t)scales + (uint64_t)(uint32_t)r * (NBLK * 4) : zsc;
        const uint32_t col_off = tile_off + (uint32_t)wave * (TK * 16);
        const uint64_t col_src = rp + 16 * wave;
        dma16(col_src, col_off);
        dma16(col_src + 128, col_off + 8 * (TK * 16));
        dma16(col_src + 256, col_off + 16 * (TK * 16));
        dma16(col_src + 384, col_off + 24 * (TK * 16));
        if (wave < 4) dma16(col_src + 512, col_off + 32 * (TK * 16));
        else dma4(sp + 4 * (wave - 4), tile_off + SC_OFF + (uint32_t)(wave - 4) * (TK * 4));
        if (wave == 0) dma4(sp + 16, tile_off + SC_OFF + 4u * (TK * 4));
    };
    // a tile by the four value waves alone (the loop: the scoring waves are the longer pole of a
    // step and a wave stalls while the memory pipeline takes its copies): wave cw copies columns
    // cw, cw + 4, .. cw + 32, scale block cw, and wave 4 also scale block 4.  The copies stand at the top
    // of a step, and what their addresses take stands in front of them: for a whole tile the lanes' offsets
    // are constants and the tile's place is a scalar (4096 queries of 128 heads over 28672 + 4096 rows:
    // 26.39 -> 26.22 ms; an address per lane takes two 64-bit multiplications a tile).
    const uint32_t lane_row = (uint32_t)lane * KDIM + 16 * cw, lane_sc = (uint32_t)lane * (NBLK * 4);
    auto share_v = [&](int t, uint32_t tile_off) {
        const uint32_t col_off = tile_off + (uint32_t)cw * (TK * 16);
        // the 64 k bytes to the lane's source are the instruction's immediate offset, which the
        // hardware also adds to the LDS address: M0 is set that much below the column
#define CWICK_P64_M0(k) "s"(col_off + (uint32_t)(4 * k) * (TK * 16) - 64u * k)
#define CWICK_P64_COL(k)                                                                                  \
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 offset:" #k "*64"         \
                 ::"v"(lane_row), "s"(rp), CWICK_P64_M0(k) : "memory")
        if ((t + 1) * TK <= n_keys) {
            const uint64_t rp = (uint64_t)(uintptr_t)rows + (uint64_t)(uint32_t)t * (TK * KDIM);
            const uint64_t sp = (uint64_t)(uintptr_t)scales + (uint64_t)(uint32_t)t * (TK * NBLK * 4);
            CWICK_P64_COL(0); CWICK_P64_COL(1); CWICK_P64_COL(2); CWICK_P64_COL(3); CWICK_P64_COL(4);
            CWICK_P64_COL(5); CWICK_P64_COL(6); CWICK_P64_COL(7); CWICK_P64_COL(8);
#undef CWICK_P64_COL
#undef CWICK_P64_M0
            auto dma4s = [&](uint64_t base, uint32_t lds_off) {
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(lane_sc), "s"(base), "s"(lds_off) : "memory");
            };
            dma4s(sp + 4 * cw, tile_off + SC_OFF + (uint32_t)cw * (TK * 4));
            if (cw == 0) dma4s(sp + 16, tile_off + SC_OFF + 4u * (TK * 4));
        } else {                                          // the group's last tile, if it is not whole
            const int r = t * TK + lane;
            const bool live = r < n_keys;
            const uint64_t rp = live ? (uint64_t)(uintptr_t)rows + (uint64_t)(uint32_t)r * KDIM : zrow;
            const uint64_t sp = live ? (uint64_t)(uintptr_t)scales + (uint64_t)(uint32_t)r * (NBLK * 4) : zsc;
#pragma clang loop unroll(disable)
            for (int k = 0; k < 9; k++) dma16(rp + 16 * cw + 64 * k, col_off + (uint32_t)(4 * k) * (TK * 16));
            dma4(sp + 4 * cw, tile_off + SC_OFF + (uint32_t)cw * (TK * 4));
            if (cw == 0) dma4(sp + 16, tile_off + SC_OFF + 4u * (TK * 4));
        }
    };
    // ---- Q for 4 x 16 heads as two E4M3 terms per 32-dim block with one E8M0 scale per head and
    // 128-dim block: unit u = 5 hq + b is prepared by wave u % 8 and parked where tile stage 2 and the
    // exchange area will be.  lane (n, g) holds head n of the block, dims 128 b + 32 g + [0, 32); the
    // rope block is one register set: lanes g < 2 hold the hi term of dims 512 + 32 g.., lanes g >= 2
    // the lo term of dims 512 + 32 (g - 2)...
    // Q travels like the tiles: copied as it is into the units' places, tile 0 behind it, and every wave
    // converts its units where they lie while tile 0 arrives; tile 1 goes out behind that.  A copy takes the
    // memory pipeline one cycle for every cache line that it touches, so a Q instruction walks along the
    // rows (four heads x 256 bytes), not across them (64 lines; the prologue took 12 000 cycles then).
    // Piece x (16 bytes) of head h sits at place x ^ h of the head's sixteen, so that the sixteen heads of
    // a fragment read come from different banks.
#pragma clang loop unroll(disable)
    for (int u = wave; u < 5 * (int)gsz; u += NWAVES) {
        const int hqu = (u * 13) >> 6, b = u - 5 * hqu;           // u / 5 for u < 20
        const uint32_t rb = rb_of((uint32_t)hqu), y = div_by(rb, nhb_inv);
        const int head0 = 16 * (int)(rb - y * nhb);
        const uint64_t base = (uint64_t)(uintptr_t)(q + (size_t)y * nh * KDIM + 128 * b);
        const uint32_t pu = lds0 + PARK + (uint32_t)u * PARK_UNIT;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int h = 4 * c + g, head = head0 + h < nh ? head0 + h : nh - 1;
            const int x = (n ^ h) & (b < 4 ? 15 : 7);             // the rope block has eight pieces: fetched twice
            dma16(base + (uint64_t)(uint32_t)head * (KDIM * 2) + (uint32_t)(16 * x), pu + (uint32_t)c * 1024);
        }
    }
    if (n_tiles > 0) {
        share(0, lds0);
        asm volatile("s_waitcnt vmcnt(5)" ::: "memory");          // a wave copies five or six pieces of a tile
    } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    {
#pragma clang loop unroll(disable)
        for (int u = wave; u < 5 * (int)gsz; u += NWAVES) {
            const uint32_t pu = lds0 + PARK + (uint32_t)u * PARK_UNIT, pr = pu + (uint32_t)lane * 16;
            u32x4 w[4];                                           // head n, pieces 4 g .. (rope: 4 (g & 1) ..)
#pragma unroll
            for (int c = 0; c < 4; c++) w[c] = LDS_AT(lds_u32x4, pu + (uint32_t)(n * 256 + (((4 * g + c) ^ n) & 15) * 16));
            u32x4 hi[2], lo[2];
            const uint32_t unit_byte = q_two_terms(w, hi, lo);
            const bool rope_lo = (u * 13 & 63) >= 4 * 13 && g >= 2;     // u % 5 == 4
#pragma unroll
            for (int c = 0; c < 2; c++) {
                LDS_AT(lds_u32x4, pr + (uint32_t)c * 1024) = rope_lo ? lo[c] : hi[c];
                LDS_AT(lds_u32x4, pr + PARK_LO + (uint32_t)c * 1024) = lo[c];
            }
            LDS_AT(lds_u32, lds0 + PARK_SC + (uint32_t)(u * 256 + lane * 4)) = unit_byte;
        }
    }
    if (n_tiles > 1) share(1, lds0 + TILE_B);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");              // tiles 0 and 1 have landed (this wave's share)
    LDS_BARRIER();

    const float c0 = p.scale * 1.44269504088896340736f;   // scores in log2 units
    // The stages rotate in scalar registers: st_val holds tile t, st_sc tile t+1, st_cp is where
    // tile t+2 goes (t % 3 as an induction variable made the compiler keep a dozen per-lane
    // addresses alive).
    uint32_t st_val = lds0 + 2 * TILE_B, st_sc = lds0, st_cp = lds0 + TILE_B;    // at t = -1
    auto rotate = [&]() {
        const uint32_t v = st_val;
        st_val = st_sc;
        st_sc = st_cp;
        st_cp = v;
        st_val = (uint32_t)__builtin_amdgcn_readfirstlane((int)st_val);
        st_sc = (uint32_t)__builtin_amdgcn_readfirstlane((int)st_sc);
        st_cp = (uint32_t)__builtin_amdgcn_readfirstlane((int)st_cp);
    };

    if (scorer) {
        // (read here and not in front of the branch: there the operands' 72 registers would be set
        // aside in the value waves' loop as well)
        i32x8 qhi[4], qlo[4], qrope;
        int qsc0 = 0, qsc1;                               // scale bytes of blocks 0..3 / of the rope block
        auto park8 = [&](uint32_t a) -> i32x8 {
            const u32x4 x = LDS_AT(lds_u32x4, a), y = LDS_AT(lds_u32x4, a + 1024);
            return (i32x8){(int)x[0], (int)x[1], (int)x[2], (int)x[3], (int)y[0], (int)y[1], (int)y[2], (int)y[3]};
        };
        const uint32_t hp = (uint32_t)hq < gsz ? (uint32_t)hq : gsz - 1;
        const uint32_t pq = lds0 + PARK + 5 * hp * PARK_UNIT + (uint32_t)lane * 16;
        const uint32_t pc = lds0 + PARK_SC + 5 * hp * 256 + (uint32_t)lane * 4;
#pragma unroll
        for (int b = 0; b < 4; b++) {
            qhi[b] = park8(pq + (uint32_t)b * PARK_UNIT);
            qlo[b] = park8(pq + (uint32_t)b * PARK_UNIT + PARK_LO);
            qsc0 |= (int)(LDS_AT(lds_u32, pc + (uint32_t)b * 256) << (8 * b));
        }
        qrope = park8(pq + 4 * PARK_UNIT);
        qsc1 = (int)LDS_AT(lds_u32, pc + 4 * 256);
        LDS_BARRIER();                                    // the park area becomes tile stage and exchange
        // Nothing the compiler has in flight may cross into the loop: its waits would also wait for
        // the copies.
        asm volatile("" : "+v"(qhi[0]), "+v"(qhi[1]), "+v"(qhi[2]), "+v"(qhi[3]), "+v"(qlo[0]), "+v"(qlo[1]), "+v"(qlo[2]), "+v"(qlo[3]), "+v"(qrope), "+v"(qsc0), "+v"(qsc1));
        float l_priv = 0.0f;                              // sum over this lane's keys of head 16 hq + n, relative to mr
        float mr = -INFINITY;                             // the reference of head 16 hq + n (the four lanes of a head agree)
        // per-lane LDS offsets inside a tile: K fragment of key block 0 (key n, columns 8 b + 2 g and
        // the next), the rope block's (columns 32 + 2 (g & 1)), this lane's four keys' scales
        const uint32_t k_off = (uint32_t)((2 * g) * (TK * 16) + n * 16);
        const uint32_t kr_off = (uint32_t)((32 + 2 * (g & 1)) * (TK * 16) + n * 16);
        // the scales of the tile's keys: lane (row g, place j) holds the scale of key
        // 16 (j / 4) + 4 g + j % 4, the key that accumulator register j % 4 of key block j / 4 holds in
        // this row: one register per dim block covers the tile (five 4-byte reads instead of twenty
        // 16-byte ones, a quarter of what the four scoring waves read from LDS per tile), and the
        // combination of the block products takes its factor from place 4 kb + i of the row
        const uint32_t sr_off = SC_OFF + (uint32_t)((16 * (n >> 2) + 4 * g + (n & 3)) * 4);
        // where this lane's four probabilities of key block kb go: keys 16 (kb & 1) + 4 g + i of half kb >> 1
        const uint32_t xp_off = (uint32_t)(((hq * 2 * 4 + (g >> 1)) * 16 + n) * 16 + 2 * (g & 1) * 4);
        const uint32_t xc_off = XC_OFF + (uint32_t)((hq * 16 + n) * 4);
        const uint32_t xf_off = XF_OFF + (uint32_t)(hq * 4);
        const int my_keys = keys_of((uint32_t)hq);        // what the wave's query sees of the slice (any sign)

#pragma clang loop unroll(disable)
        for (int t = 0; t < n_tiles; t++) {
            {
                // ---- scores S^T[key][head] for all 64 keys, heads 16 hq.. of tile t ----
                const uint32_t tb = st_sc;
                const uint32_t xn = lds0 + X_OFF + (uint32_t)(t & 1) * XCH_B;
                f32x4 S[4];
                float rsc[NBLK];
#pragma unroll
                for (int b = 0; b < NBLK; b++) rsc[b] = LDS_AT(lds_f32, tb + sr_off + (uint32_t)b * (TK * 4));
                // Fragment j = 5 kb + b (b = 4: the rope block).  Its MFMAs (hi and lo term, or the one
                // rope instruction) are issued from assembly in a fixed order, its block product is
                // folded into S three fragments later: between an MFMA and the statement that reads its
                // result lie the MFMAs and folds of three other fragments (fifteen instructions or
                // more, where an 8-pass MFMA asks for eleven), and a lo term accumulates into the
                // registers its hi term wrote.
                const uint32_t kbase = tb + k_off, krbase = tb + kr_off;
                auto kfrag = [&](int j) -> i32x8 {
                    const int kb = j / 5, b = j % 5;
                    const uint32_t a = (b < 4 ? kbase + (uint32_t)(8 * b) * (TK * 16) : krbase) + (uint32_t)kb * 256u;
                    const u32x4 k0 = LDS_AT(lds_u32x4, a);
                    const u32x4 k1 = LDS_AT(lds_u32x4, a + TK * 16);
                    return (i32x8){(int)k0[0], (int)k0[1], (int)k0[2], (int)k0[3], (int)k1[0], (int)k1[1], (int)k1[2], (int)k1[3]};
                };
                const int one_scales = 0x7F7F7F7F;
#define CWICK_P64_PAIR(A, K, QH, QL, SEL)                                                                         \
    asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, 0, %4, %5 " SEL "\n\t"                             \
                 "v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %3, %0, %4, %5 " SEL                                    \
                 : "=&v"(A) : "v"(K), "v"(QH), "v"(QL), "v"(one_scales), "v"(qsc0))
                f32x4 acc[4];
                i32x8 kfr[3];
                kfr[0] = kfrag(0);
                kfr[1] = kfrag(1);
#pragma unroll
                for (int j = 0; j < 23; j++) {
                    if (j < 20) {
                        const int b = j % 5;
                        if (j + 2 < 20) kfr[(j + 2) % 3] = kfrag(j + 2);
                        switch (b) {
                            case 0: CWICK_P64_PAIR(acc[j % 4], kfr[j % 3], qhi[0], qlo[0], "op_sel:[0,0,0] op_sel_hi:[0,0,0]"); break;
                            case 1: CWICK_P64_PAIR(acc[j % 4], kfr[j % 3], qhi[1], qlo[1], "op_sel:[0,1,0] op_sel_hi:[0,0,0]"); break;
                            case 2: CWICK_P64_PAIR(acc[j % 4], kfr[j % 3], qhi[2], qlo[2], "op_sel:[0,0,0] op_sel_hi:[0,1,0]"); break;
                            case 3: CWICK_P64_PAIR(acc[j % 4], kfr[j % 3], qhi[3], qlo[3], "op_sel:[0,1,0] op_sel_hi:[0,1,0]"); break;
                            default:
                                asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, 0, %3, %4 op_sel:[0,0,0] op_sel_hi:[0,0,0]"
                                             : "=&v"(acc[j % 4]) : "v"(kfr[j % 3]), "v"(qrope), "v"(one_scales), "v"(qsc1));
                                break;
                        }
                    } else {
                        asm volatile("s_nop 3" ::: "memory");          // the last three folds have no MFMAs behind them
                    }
                    if (j >= 3) {
                        const int f = j - 3, kb = f / 5, b = f % 5;
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            float d = S[kb][i];
                            scaled_by_row_lane(d, rsc[b], acc[f % 4][i], 4 * kb + i, b == 0);
                            S[kb][i] = d;
                        }
                    }
                }
#undef CWICK_P64_PAIR
                // positions past the query's last key (only in its last tile, and in a tile that only
                // later queries of the group reach; the empty statement keeps this a branch: as sixteen
                // selects it would run in every step)
                const int tail_keys = my_keys - t * TK;
                if (tail_keys < TK) {
                    asm volatile("" ::: "memory");
#pragma unroll
                    for (int kb = 0; kb < 4; kb++)
#pragma unroll
                        for (int i = 0; i < 4; i++)
                            if (16 * kb + 4 * g + i >= tail_keys) S[kb][i] = -INFINITY;
                }
                float lmax = vmax3(S[0][0], S[0][1], vmax(S[0][2], S[0][3]));
#pragma unroll
                for (int kb = 1; kb < 4; kb++) lmax = vmax3(lmax, S[kb][0], vmax3(S[kb][1], S[kb][2], S[kb][3]));
                lmax *= c0;                                   // S stays unscaled: c0 > 0 goes into the exponent's multiply-add
                const bool moves = __any(lmax > mr + LAZY);   // rare after the first tiles: only then the lanes of a head confer
                if (moves) {
                    lmax = xor16_max(lmax);
                    lmax = xor32_max(lmax);
                    const float m_new = lmax > mr + LAZY ? lmax : mr;
                    const float cf = (mr == -INFINITY || m_new == mr) ? 1.0f : __builtin_amdgcn_exp2f(mr - m_new);
                    l_priv *= cf;
                    mr = m_new;
                    LDS_AT(lds_f32, xn + xc_off) = cf;        // the four lanes of a head write the same word
                }
                const float m_use = mr == -INFINITY ? 0.0f : mr;
                float lsum = 0.0f;
#pragma unroll
                for (int kb = 0; kb < 4; kb++) {
                    f32x4 P;
#pragma unroll
                    for (int i = 0; i < 4; i++) P[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(S[kb][i], c0, -m_use));
                    lsum += (P[0] + P[1]) + (P[2] + P[3]);
                    u32x2 d;
                    d[0] = pack_f16_rne(P[0], P[1]);
                    d[1] = pack_f16_rne(P[2], P[3]);
                    // [hq][kb >> 1][2 (kb & 1) + (g >> 1)][n][2 (g & 1) ..]
                    LDS_AT(lds_u32x2, xn + xp_off + (uint32_t)(((kb >> 1) * 4 + 2 * (kb & 1)) * 256)) = d;
                }
                l_priv += lsum;
                LDS_AT(lds_u32, xn + xf_off) = moves ? 1u : 0u;
            }
            LDS_BARRIER();
            rotate();
        }
        LDS_BARRIER();                                    // the value waves' last step

        // ---- the sums of the scoring role meet in LDS (the exchange area is free now) ----
        float *lsum = reinterpret_cast<float *>(&sm.x[0]);            // [16-head block][head], then the references
        float ls = xor16_sum(l_priv);
        ls = xor32_sum(ls);
        if (g == 0) {
            lsum[hq * 16 + n] = ls;
            lsum[64 + hq * 16 + n] = mr;
        }
        LDS_BARRIER();
    } else {
        LDS_BARRIER();                                    // the scoring waves have their Q
        f32x4 oacc[NHQ][8];                               // [16-head block][dim block]: dims 128 cw + 16 j + 4 g + i, head n
#pragma unroll
        for (int h = 0; h < NHQ; h++)
#pragma unroll
            for (int j = 0; j < 8; j++) oacc[h][j] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
        int e_run = E_NONE;                               // 2^e_run is above every scale of this wave's block seen so far
        uint32_t thr_bits = 0u;                           // bits of 2^e_run: a scale whose bits reach them does not fit
        float wfac = 0.0f;                                // 2^(WEXP - e_run)
        __builtin_amdgcn_s_setprio(3);
        // transpose-read addressing for V^T: lane i of 16-lane group g supplies key 8 g + (i >> 1),
        // bytes 8 (i & 1) .. +7 of the sixteen-byte column
        const uint32_t tr_off = (uint32_t)((8 * cw) * (TK * 16) + (8 * g + (n >> 1)) * 16 + 8 * (n & 1));
        // the two scales this lane turns into a pair of factors (see the loop)
        const uint32_t sv_off = SC_OFF + (uint32_t)(cw * (TK * 4) + (32 * ((n & 7) >> 2) + 8 * g + 2 * (n & 3)) * 4);
        // the probabilities of this lane's slots: [16-head block][key half][g][n][4 dwords]
        const uint32_t pw_off = (uint32_t)((g * 16 + n) * 16);
        const uint32_t xcl_off = XC_OFF + (uint32_t)(n * 4);
        const int keys_lo = keys_of(0);                   // of the group's first query
        asm volatile("" ::: "memory");
        LDS_BARRIER();                                    // tile 0 is scored
        rotate();
#pragma clang loop unroll(disable)
        for (int t = 0; t < n_tiles; t++) {
            if (t + 2 < n_tiles) share_v(t + 2, st_cp);   // the stage tile t-1 left at the last barrier
            {
                // ---- values O^T[dim][head] += V^T W^T for dims 128 cw.., all 64 heads, tile t ----
                const uint32_t tb = st_val;
                const uint32_t xb = lds0 + X_OFF + (uint32_t)(t & 1) * XCH_B;
                // The sixteen lanes of a row share their contraction slots (keys 8 g .. 8 g + 7 of each
                // half), so a row needs eight fp16 pairs of scale factors per tile: lane (g, n) reads
                // the two scales of pair n & 7 (half (n & 7) >> 2, keys 8 g + 2 (n & 3) and the next),
                // forms that one pair, and every lane takes the eight pairs out of the row by DPP.
                f32x2 sv = LDS_AT(lds_f32x2, tb + sv_off);
                const u32x4 fl = LDS_AT(lds_u32x4, xb + XF_OFF);
                // SPAN: keys of the tile that every query of the group sees; the few behind them are added
                // by themselves, to the queries that see them and to no other
                const int vis = keys_lo - t * TK;
                if (SPAN) {
                    const int k_lane = 32 * ((n & 7) >> 2) + 8 * g + 2 * (n & 3);
                    sv[0] = k_lane < vis ? sv[0] : 0.0f;
                    sv[1] = k_lane + 1 < vis ? sv[1] : 0.0f;
                }
                // normaliser of the fp16 weights: a power of two above every scale seen so far (it
                // only grows, and only then the lanes confer).  Scales are compared as integers:
                // they are positive, and a negative or NaN scale has the larger bit pattern too.
                float ecorr = 1.0f;
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
                u32x4 sw[2];                              // scale * 2^(WEXP - e_run) of the slots' keys, fp16 pairs
                sw[0][0] = row_place<0>(my_pair);
                sw[0][1] = row_place<1>(my_pair);
                sw[0][2] = row_place<2>(my_pair);
                sw[0][3] = row_place<3>(my_pair);
                sw[1][0] = row_place<4>(my_pair);
                sw[1][1] = row_place<5>(my_pair);
                sw[1][2] = row_place<6>(my_pair);
                sw[1][3] = row_place<7>(my_pair);
                const uint32_t any_moved = fl[0] | fl[1] | fl[2] | fl[3];
                if (__builtin_amdgcn_readfirstlane(any_moved) != 0u || ecorr != 1.0f) {
                    // a scoring wave moved a reference in this tile (or the weights' normaliser
                    // grew): the accumulators so far shrink to the new units
#pragma unroll
                    for (int h = 0; h < NHQ; h++) {
                        float c = ecorr;
                        if (__builtin_amdgcn_readfirstlane(fl[h]) != 0u) c *= LDS_AT(lds_f32, xb + xcl_off + (uint32_t)(h * 64));
#pragma unroll
                        for (int j = 0; j < 8; j++) oacc[h][j] *= c;
                    }
                }
                if (SPAN && vis < TK) {
                    // keys that only the group's later queries see (at most three of them): one fp32
                    // multiply-add per key and value
                    if (e_run == E_NONE) {                // nothing has set the units yet
                        e_run = WEXP;
                        thr_bits = __builtin_bit_cast(uint32_t, pow2i(e_run));
                        wfac = 1.0f;
                    }
                    for (int k = vis > 0 ? vis : 0; k < TK && t * TK + k < n_keys; k++) {
                        const float ws = LDS_AT(lds_f32, tb + SC_OFF + (uint32_t)((cw * TK + k) * 4)) * wfac;
                        f32x4 v[8];
#pragma unroll
                        for (int j = 0; j < 8; j++) {
                            const uint32_t d = LDS_AT(lds_u32, tb + (uint32_t)((8 * cw + j) * (TK * 16) + k * 16 + 4 * g));
                            const f32x2 lo = e4m3x2_to_f32<false>(d), hi = e4m3x2_to_f32<true>(d);
                            v[j] = (f32x4){lo[0], lo[1], hi[0], hi[1]} * ws;
                        }
#pragma unroll
                        for (int h = 0; h < NHQ; h++) {
                            if (t * TK + k >= keys_of(h)) continue;
                            // the probability of key k: [h][k / 32][(k % 32) / 8][n][half k % 8]
                            const uint32_t pd = LDS_AT(lds_u32, xb + (uint32_t)((((h * 2 + (k >> 5)) * 4 + ((k & 31) >> 3)) * 16 + n) * 16 + ((k & 7) >> 1) * 4));
                            const f16x2 pp = __builtin_bit_cast(f16x2, pd);
                            const float pk = (float)((k & 1) ? pp[1] : pp[0]);
#pragma unroll
                            for (int j = 0; j < 8; j++)
#pragma unroll
                                for (int i = 0; i < 4; i++) oacc[h][j][i] = __builtin_fmaf(v[j][i], pk, oacc[h][j][i]);
                        }
                    }
                    // what they are has been used: it may not reach an earlier query through its zero
                    // weight (a NaN would).  Nobody else reads these columns of this tile any more.
                    for (int k = vis > 0 ? vis : 0; k < TK && t * TK + k < n_keys; k++)
                        if (lane < 8) LDS_AT(lds_u32x4, tb + (uint32_t)((8 * cw + lane) * (TK * 16) + k * 16)) = (u32x4){0u, 0u, 0u, 0u};
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                }
                // Fragment q = 8 kh + j (key half, dim block) of V^T is requested four fragments ahead of
                // its products, into the registers of the fragment just converted: a fragment's four
                // products cover a quarter of its own latency.
                const uint32_t va0 = tb + tr_off;
                auto vfrag = [&](int q) -> i32x2 {
                    return __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_i32x2 *)(size_t)(va0 + (uint32_t)((q & 7) * (TK * 16) + (q >> 3) * (32 * 16))));
                };
                u32x4 pw[2][NHQ];                         // the tile's weights, per key half and 16-head block
                i32x2 vt[4];
#pragma unroll
                for (int h = 0; h < NHQ; h++) pw[0][h] = LDS_AT(lds_u32x4, xb + pw_off + (uint32_t)(h * 2048));
#pragma unroll
                for (int q = 0; q < 4; q++) vt[q] = vfrag(q);
#pragma unroll
                for (int h = 0; h < NHQ; h++) pw[1][h] = LDS_AT(lds_u32x4, xb + pw_off + (uint32_t)(h * 2048 + 1024));
#pragma unroll
                for (int q = 0; q < 16; q++) {
                    const int kh = q >> 3;
                    const i32x2 v2 = vt[q & 3];
                    u32x4 vh;
                    vh[0] = e4m3x2_to_f16x2<false>((uint32_t)v2[0]);
                    vh[1] = e4m3x2_to_f16x2<true>((uint32_t)v2[0]);
                    vh[2] = e4m3x2_to_f16x2<false>((uint32_t)v2[1]);
                    vh[3] = e4m3x2_to_f16x2<true>((uint32_t)v2[1]);
                    const f16x8 va = __builtin_bit_cast(f16x8, vh);
                    if (q + 4 < 16) vt[q & 3] = vfrag(q + 4);
#pragma unroll
                    for (int h = 0; h < NHQ; h++) {
                        if ((q & 7) == 0)
#pragma unroll
                            for (int d = 0; d < 4; d++) pw[kh][h][d] = mul_f16x2(pw[kh][h][d], sw[kh][d]);
                        oacc[h][q & 7] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, __builtin_bit_cast(f16x8, pw[kh][h]), oacc[h][q & 7], 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            // tile t+2, copied by the value waves during this step, is scored in the next one
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            LDS_BARRIER();
            rotate();
        }

        const float *lsum = reinterpret_cast<const float *>(&sm.x[0]);
        LDS_BARRIER();
        // ---- every value wave owns its dims: write the result, or the slice's partial ----
        const float unit_f = e_run == E_NONE ? 0.0f : pow2i(e_run - WEXP);   // the accumulators are in units of 2^(e_run - WEXP)
#pragma clang loop unroll(disable)
        for (int h = 0; h < (int)gsz; h++) {
            const float L = lsum[h * 16 + n];
            if (!sliced) {
                const uint32_t rb = gsz * grp + h, y = div_by(rb, nhb_inv);
                // Through the wave's own stretch of LDS (the tiles are done with), so that a store
                // writes 512 bytes of two heads and not 64 of sixteen, whose rows are 2 KB apart and
                // meet in two channels of the L2.
                const float fin = L > 0.0f ? unit_f / L : 0.0f;
                const uint32_t ob = lds0 + (uint32_t)cw * (16 * 528), ow = ob + (uint32_t)(n * 528 + g * 16);
#pragma unroll
                for (int j = 0; j < 8; j++)
                    LDS_AT(lds_f32x4, ow + (uint32_t)(64 * j)) = oacc[0][j] * fin;   // register i <-> dim 16 (8 cw + j) + 4 g + i
                if (rb < n_rb) {
                    const int head0 = 16 * (int)(rb - y * nhb) + (lane >> 5);
                    float *dst = p.out + ((size_t)y * nh + head0) * VDIM + 128 * cw + 4 * (lane & 31);
                    const uint32_t orow = ob + (uint32_t)((lane >> 5) * 528 + (lane & 31) * 16);
                    f32x4 v[8];
#pragma unroll
                    for (int k = 0; k < 8; k++) v[k] = LDS_AT(lds_f32x4, orow + (uint32_t)(2 * k * 528));
                    const int rows_left = nh - head0;           // (a scalar branch for whole blocks: eight predicated stores are slower)
                    if (__all(rows_left > 14)) {
#pragma unroll
                        for (int k = 0; k < 8; k++) *(f32x4 *)(dst + 2 * k * VDIM) = v[k];
                    } else {
#pragma unroll
                        for (int k = 0; k < 8; k++)
                            if (2 * k < rows_left) *(f32x4 *)(dst + 2 * k * VDIM) = v[k];
                    }
                }
            } else {
                // The layout and the write-through stores of mla_roles.hip's partials, but the accumulators as
                // they are: the sums of an uncut chunk stay in fp32 from the first product to the output, and
                // so do those that meet in the merge.
                const size_t pb = ((size_t)grp * n_slices + slice) * gsz + h;
                float *pq = p.part_acc + ((pb * (VDIM / 16) + 8 * cw) * 64 + lane) * 4;   // [dim block][lane][4]
#pragma unroll
                for (int j = 0; j < 8; j++) store_through16(pq + j * 256, __builtin_bit_cast(u32x4, oacc[0][j]));
                if (g == 0)
                    *(f32x4 *)(p.part_ml + ((pb * 4 + cw) * 16 + n) * 4) =
                        (f32x4){lsum[64 + h * 16 + n] * 0.69314718055994530942f, L, unit_f, 0.0f};
            }
            // the next row block moves up: one copy of the code above serves the four
#pragma unroll
            for (int m = 0; m + 1 < NHQ; m++)
#pragma unroll
                for (int j = 0; j < 8; j++) oacc[m][j] = oacc[m + 1][j];
        }
    }
}

}  // namespace

int launch_mla_prefill(const uint8_t *rows, const float *scales, int64_t pos0, int64_t n,
                       const uint16_t *q, int n_heads, float scale, float *out, hipStream_t s) {
    CWICK_REQUIRE(rows && scales && q && out, "mla_prefill: null pointer");
    CWICK_REQUIRE(n_heads >= 1 && n_heads <= 128, "mla_prefill: n_heads %d (1..128)", n_heads);
    CWICK_REQUIRE(pos0 >= 0 && n >= 1 && pos0 + n <= ((int64_t)1 << 31) - 1 && n <= (1 << 22),
                  "mla_prefill: pos0 %lld n %lld", (long long)pos0, (long long)n);
    CWICK_REQUIRE(scale > 0.0f && scale < INFINITY, "mla_prefill: scale must be positive");
    CWICK_REQUIRE((uintptr_t)rows % 16 == 0 && (uintptr_t)q % 16 == 0 && (uintptr_t)out % 16 == 0,
                  "mla_prefill: rows, q and out must be 16-byte aligned");
    static std::once_flag attr_once;
    static hipError_t attr_err = hipSuccess;
    const size_t smem = SMEM_BYTES;
    std::call_once(attr_once, [&] {
        attr_err = hipFuncSetAttribute((const void *)mla_prefill64_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
        if (attr_err == hipSuccess)
            attr_err = hipFuncSetAttribute((const void *)mla_prefill64_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    });
    CWICK_HIP_CALL(attr_err);
    WideRest p{};
    p.scale = scale; p.out = out;
    const uint32_t nhb = (uint32_t)(n_heads + 15) / 16, n_rb = (uint32_t)n * nhb;               // below 2^25
    WidePlan plan = plan_wide((int64_t)n_rb, (pos0 + 1 + TK - 1) / TK, (pos0 + n + TK - 1) / TK, num_cus());
    if (plan.whole < plan.groups) {
        const size_t blocks = (size_t)(plan.groups - plan.whole) * plan.slices * plan.gsz;
        const size_t acc_b = blocks * 16 * VDIM * sizeof(float);
        char *ws = (char *)workspace_if_free(s, acc_b + blocks * 4 * 16 * 4 * sizeof(float));
        p.part_acc = (float *)ws;
        p.part_ml = (float *)(ws + acc_b);
        // no room for partials (a stream that is being captured and has not run the shape before): uncut
        if (!ws) plan = WidePlan{NHQ, (n_rb + NHQ - 1) / NHQ, (n_rb + NHQ - 1) / NHQ, 1, 0.0f};
    }
    const uint32_t n_rest = plan.groups - plan.whole;
    {
        ProfKernel pk(CWICK_HIP_PROF_MLA_PREFILL, s);
        pk.launch(nhb % plan.gsz == 0 ? mla_prefill64_kernel<false> : mla_prefill64_kernel<true>, dim3(plan.whole + n_rest * plan.slices),
                  dim3(THREADS), smem, q, rows, scales, (int)pos0, (uint32_t)n_heads | plan.gsz << 8, div_inverse(nhb), n_rb, plan.whole,
                  n_rest, plan.slices, div_inverse(plan.slices), p);
    }
    CWICK_HIP_CALL(hipGetLastError());
    if (n_rest)
        return launch_mla_merge((const f32x4 *)p.part_acc, p.part_ml, (int)plan.slices, (int)n_rest, (int)plan.gsz, (int)nhb, (int64_t)n_rb,
                                n_heads, nullptr, out, CWICK_HIP_PROF_MLA_MERGE, s);
    return 1;
}

}  // namespace cwick
