// common.hpp -- shared declarations of libcwick_hip.so (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <stdint.h>
#include <stddef.h>

#include <initializer_list>

#include "../../include/cwick_hip.h"
#include "band_counter.hpp"

namespace cwick {

// ---- error reporting -------------------------------------------------------
// Every extern "C" entry point returns 0 ("declined") after recording why.
void set_error(const char *fmt, ...) __attribute__((format(printf, 1, 2)));
void clear_error();
bool hip_ok(hipError_t e, const char *what);   // records the error text on failure

#define CWICK_REQUIRE(cond, ...)            \
    do {                                    \
        if (!(cond)) {                      \
            ::cwick::set_error(__VA_ARGS__); \
            return 0;                       \
        }                                   \
    } while (0)

#define CWICK_HIP_CALL(expr)                          \
    do {                                              \
        if (!::cwick::hip_ok((expr), #expr)) return 0; \
    } while (0)

// ---- runtime ---------------------------------------------------------------
bool backend_ready();                       // device 0 is up and selected
int num_cus();
// Grow-only scratch keyed by stream and slot.  A call's buffer stays valid for the kernels it
// enqueues (and for graphs captured from them) until the stream is released: growing allocates
// a new buffer and retires the old one, it neither frees nor waits.  Returns null (reason
// recorded) when it would have to allocate while the stream is being captured.
// Slot WS_NESTED belongs to launchers that other launchers call with operands in slot WS_MAIN
// (the top-k select inside the block selections).
constexpr int WS_MAIN = 0, WS_NESTED = 1, WS_SLOTS = 2;
// A launcher asks for what any smaller call of its kind would need too, so that a stream that has run a
// shape has room for the smaller ones under capture.
void *workspace(hipStream_t s, size_t bytes, int slot = WS_MAIN);
// The same for launchers that can do without: null, and nothing recorded.
void *workspace_if_free(hipStream_t s, size_t bytes);
// Where a kernel reports to the host that its results are there: workgroup i writes `epoch` to flags[i]
// (host memory) when its stores are through.  The launcher says how many workgroups do.
struct HostFlags {
    uint32_t *flags;
    uint32_t epoch;
    int count;
};
constexpr int HOST_FLAGS_MAX = 1024;
uint32_t *ticket_counters(hipStream_t s);   // 64 dwords per stream, zero between kernels; null under capture if not there yet
uint32_t *ticket_counters_if_free(hipStream_t s);   // the same, and nothing recorded

// Phase timer: brackets the launches made while it is alive with two events on
// `s` when profiling is enabled; does nothing (and records nothing) otherwise.
struct ProfScope {
    ProfScope(int which, hipStream_t s);
    ~ProfScope();
    int which;
    hipStream_t stream;
    void *slot;
};

// Phase timer of exactly one kernel: when profiling is enabled the launch goes through
// hipExtLaunchKernelGGL with a start and a stop event that the runtime binds to the dispatch
// itself, so their difference is the kernel's own duration (what a kernel trace reports), not
// the dispatch latency that an event pair recorded around the launch includes.  Otherwise an
// ordinary launch, no events.
struct ProfKernel {
    ProfKernel(int which, hipStream_t s);
    ~ProfKernel();
    template <typename... KArgs, typename... Args>
    void launch(void (*kernel)(KArgs...), dim3 grid, dim3 block, size_t smem, Args... args) {
        if (a) {
            hipExtLaunchKernelGGL(kernel, grid, block, (uint32_t)smem, stream, a, b, 0u, static_cast<KArgs>(args)...);
            bound = true;
        } else {
            kernel<<<grid, block, smem, stream>>>(static_cast<KArgs>(args)...);
        }
    }
    int which;
    hipStream_t stream;
    hipEvent_t a = nullptr, b = nullptr;
    bool bound = false;
};

// ---- kernel launchers (one per .hip file) ----------------------------------
int launch_gqa_decode(const uint16_t *k, const uint16_t *v, int64_t n_keys, int n_kv_heads,
                      int head_dim, const uint16_t *q, int n_heads, float scale, float *out,
                      hipStream_t s, const int32_t *sel = nullptr, int64_t n_rows = 0, HostFlags *done = nullptr);
int launch_gqa_prefill(const uint16_t *k, const uint16_t *v, int64_t pos0, int64_t n,
                       int n_kv_heads, int head_dim, const uint16_t *q, int n_heads,
                       float scale, float *out, hipStream_t s);
int launch_mla_decode(const uint8_t *rows, const float *scales, int64_t row_bstride,
                      int64_t scale_bstride, int64_t n_rows, int batch, const int32_t *sel, int64_t n_list,
                      const uint16_t *q, int n_heads, float scale, const float *sink, float *out,
                      hipStream_t s, bool fixed_scratch = false);
int launch_mla_prefill(const uint8_t *rows, const float *scales, int64_t pos0, int64_t n,
                       const uint16_t *q, int n_heads, float scale, float *out, hipStream_t s);
int launch_indexer_scores(const uint8_t *keys, const float *kscale, int64_t key_bstride,
                          int64_t kscale_bstride, int batch, int64_t n_keys,
                          const uint16_t *q_idx, const float *w, int n_idx_heads, int mode,
                          float *scores, hipStream_t s);
// ---- fused select: approximate scores with an error band, exact scores for the keys inside it
// (indexer_band.hip).  One of these per batch row, in the workspace:
struct IndexerBandRow {
    uint32_t n_cand;      // keys inside the band (may exceed the list's capacity)
    uint32_t fallback;    // the band could not be formed (bound not finite, NaN threshold)
    uint32_t octave;      // the lowest of the octaves that the row's counters resolve (band_counter)
    uint32_t pad[29];     // a row to a 128-byte line: the workgroups of different rows add to n_cand at the same time
};
constexpr int CWICK_INDEXER_BAND_CAP = 4096;   // candidate list entries per row
// Keys per workgroup (= per slot of bounds and counts) of the approximate kernel: 2048, or fewer where that
// leaves compute units without one (a workgroup takes 5 us and 1.2 per 256 keys; what the select adds up of a
// row grows with its slots, so at most 128).  With the attention, rows of 64K keys: one 44.7 us with 2048, 38.6
// with 512; two 48.3, 41.1; four 49.2, 46.6 with 1024; eight of 16000 49.3, 43.9 with 512.
constexpr int CWICK_INDEXER_APPROX_KEYS = 2048, CWICK_INDEXER_APPROX_SLOTS = 128;
inline int indexer_approx_keys(int64_t n_keys, int batch) {
    for (int keys : {512, 768, 1024, 1536}) {
        const int64_t slots = (n_keys + keys - 1) / keys;
        if (slots * batch <= num_cus() && slots <= CWICK_INDEXER_APPROX_SLOTS) return keys;
    }
    return CWICK_INDEXER_APPROX_KEYS;
}
inline int indexer_approx_slots(int64_t n_keys, int batch) {
    const int keys = indexer_approx_keys(n_keys, batch);
    return (int)((n_keys + keys - 1) / keys);
}
int launch_indexer_approx(const uint8_t *keys, const float *kscale, int64_t key_bstride,
                          int64_t kscale_bstride, int batch, int64_t n_keys, const uint16_t *q_idx,
                          const float *w, int n_idx_heads, float *scores, float *beta_slots,
                          IndexerBandRow *rows, uint32_t *digits, hipStream_t s);
// What the approximate kernel leaves for the select, per row and workgroup (slot): how many of its scores
// each of 4096 counters has (16-bit counts; band_counter), and each sixteen of them together.
constexpr int CWICK_BAND_DIGITS = 256 + 4096 / 2;         // dwords per slot
// (of a call: as much as any call of fewer rows or keys needs)
inline size_t indexer_band_digits_dwords(int64_t n_keys, int batch) {
    const size_t slots = (size_t)indexer_approx_slots(n_keys, batch) * batch, few = (size_t)num_cus();
    return (slots > few ? slots : few) * CWICK_BAND_DIGITS;
}
__host__ __device__ inline bool indexer_band_failed(const IndexerBandRow &r, int cap) {
    return r.fallback != 0u || r.n_cand > (uint32_t)cap;
}
// shapes the banded path takes: rows that the many-workgroup top-k handles, k < n
// The banded select is four launches, about the same for any row; every key scored exactly and one
// workgroup's select take 5.05 us per million key-head pairs of the batch and 0.37 per 1024 keys of a row: the
// difference is 15.8 less than these (26 shapes on either side of the line, off by 2.5 us at most).  With the
// attention, 64 heads: one row of 24000 keys 33.7 us against 33.8, of 28000 39.7 against 34.0; 2 x 14000 32.1 against
// 34.0, 2 x 18000 38.3 against 35.0; 4 x 8300 35.1 against 36.4, 4 x 13000 42.5 against 36.4; 8 x 8300 51.4 against 41.9.
inline bool indexer_band_applies(int64_t n_keys, int64_t k, int n_idx_heads, int batch) {
    return n_keys > 6144 && n_keys <= 131072 && k < n_keys && n_idx_heads >= 1 && n_idx_heads <= 64 &&
           5.05e-6 * (double)(n_keys * batch * n_idx_heads) + 3.7e-4 * (double)n_keys > 15.8;
}
// indexer and top-k in one: `scores` is scratch (its contents afterwards are not scores), the
// selected indices of every row go to out_idx[batch][k] in ascending order
int launch_indexer_banded(const uint8_t *keys, const float *kscale, int64_t key_bstride,
                          int64_t kscale_bstride, int batch, int64_t n_keys, const uint16_t *q_idx,
                          const float *w, int n_idx_heads, int64_t k, float *scores, int32_t *out_idx,
                          hipStream_t s);
// top-k machinery on approximate scores: finds the counter that T is in from the approximate kernel's counts, then
// patches the scores (+inf / -inf / kept) and lists the keys that may lie on either side.
size_t topk_mw_workspace_bytes(int batch, int64_t n);
int launch_topk_band_classify(float *scores, int batch, int64_t n, int64_t k, const uint32_t *digits,
                              const float *beta_slots, int n_beta, int32_t *cand, int cap,
                              IndexerBandRow *rows, uint32_t *hi_count, hipStream_t s);
// The end of the banded select, after the candidates have their exact scores: ranks the
// candidates, writes the selected indices of every row that fitted the band, and runs the
// plain select for the rows that did not (their scores are the exact kernel's by then).
// `scores` is only read.
// hi_count: [batch][64] dwords, filled by launch_topk_band_classify.
// cand_score: [batch][cap], the exact score of every list entry (what the rescoring wrote).
int launch_topk_band_finish(float *scores, int batch, int64_t n, int64_t k, const int32_t *cand,
                            const float *cand_score, int cap, const IndexerBandRow *rows, uint32_t *hi_count,
                            int32_t *out_idx, hipStream_t s);
int launch_topk(const float *scores, int batch, int64_t n, int64_t k, int32_t *out_idx,
                hipStream_t s);
int launch_quant_latent(const float *rows, int64_t n, uint8_t *out_rows, float *out_scales,
                        hipStream_t s);
int launch_quant_ikeys(const float *rows, int64_t n, uint8_t *out_rows, float *out_scales,
                       hipStream_t s);
int launch_narrow_bf16(const float *src, int64_t n, uint16_t *dst, hipStream_t s);
// n floats (a multiple of four) to each of two arrays; copies of whole sixteen-byte pieces
int launch_narrow_pair(const float *src_a, const float *src_b, int64_t n, uint16_t *dst_a, uint16_t *dst_b, HostFlags *done,
                       hipStream_t s);
int launch_stage_copy(const void *src, void *dst, size_t bytes, HostFlags *done, hipStream_t s);
int launch_mla_absorb(const uint16_t *kvb_w, const float *q, int64_t q_stride, int batch, int n_heads,
                      int q_dim, int nope, int rope, int kv_dim, int kv_lora, uint16_t *q_abs, hipStream_t s);
int launch_mla_expand(const uint16_t *kvb_w, const float *c_acc, int batch, int n_heads, int nope, int vdim,
                      int kv_dim, int kv_lora, float *out, hipStream_t s);
int launch_gqa_prepare(const float *q_proj, int64_t q_head_stride, const float *k_proj, const float *v_proj,
                       int64_t n, int64_t pos0, int n_heads, int n_kv_heads, int head_dim, const float *q_norm,
                       const float *k_norm, float eps, const float *rope_cos, const float *rope_sin, int rotary_dim,
                       uint16_t *q_out, uint16_t *k_cache, uint16_t *v_cache, hipStream_t s);
int launch_ikeys_pool(const float *tail_k, const float *tail_g, const uint16_t *ape, const float *knw, const float *knb,
                      float eps, int kpool, int64_t n_pools, uint8_t *out_rows, float *out_scales, float *out_f32,
                      hipStream_t s);
int launch_candidate_select(const float *scores, int batch, int64_t n, int block, int64_t topk_blocks, uint8_t *cand,
                            hipStream_t s);
int launch_mm_select(const uint16_t *idx_keys, const float *iq, int batch, int64_t limit0, int index_heads,
                     int index_dim, int block, int keep_blocks, float *scores, int64_t score_stride,
                     int32_t *blk_out, int32_t *sel, int64_t max_sel, int32_t *n_sel, hipStream_t s);
int launch_candidate_apply(float *scores, const uint8_t *cand, int batch, int64_t n, hipStream_t s);
int launch_glm_select(const float *scores, int batch, int64_t n_comp, int64_t npos, int kpool, int64_t topk,
                      int strict, int32_t *sel, int64_t max_sel, int32_t *n_sel, hipStream_t s);
int launch_dequant_latent(const uint8_t *rows, const float *scales, int64_t n, float *out, hipStream_t s);
int launch_dequant_ikeys(const uint8_t *rows, const float *scales, int64_t n, float *out, hipStream_t s);
int launch_widen_bf16(const uint16_t *src, int64_t n, float *dst, hipStream_t s);
int launch_e4m3_table(float *out256_dev, hipStream_t s);
int launch_lane_ops(const uint32_t *in64_dev, uint32_t *out832_dev, hipStream_t s);
int run_probe_hbm_read(size_t bytes, int reps, double *gbps);
int run_probe_mfma(int kind, int reps, double *tflops);

// ---- device helpers ---------------------------------------------------------
// order-preserving 32-bit key of a score for the radix select: larger score, larger key; NaN
// sorts below everything (key 0), -0.0 equals +0.0, and no number maps to 0
__device__ __forceinline__ uint32_t topk_key(float f) {
    const uint32_t u = __builtin_bit_cast(uint32_t, f + 0.0f);        // -0.0 + 0.0 is +0.0
    const uint32_t key = u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
    return f != f ? 0u : key;                                         // (only a NaN's bits would give key 0)
}
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;

// partials of mla_roles.hip's layout, [group][split][16-row block], 16-bit fixed point or fp32, into out: row block
// rb = n_hb16 * group + block is heads 16 (rb % nhb) .. of query rb / nhb; blocks from n_rb on are not there
int launch_mla_merge(const u32x2 *part_acc, const float *part_ml, int n_splits, int n_groups, int n_hb16, int nhb,
                     int64_t n_rb, int nh, const float *sink, float *out, int prof, hipStream_t s);
int launch_mla_merge(const f32x4 *part_acc, const float *part_ml, int n_splits, int n_groups, int n_hb16, int nhb,
                     int64_t n_rb, int nh, const float *sink, float *out, int prof, hipStream_t s);

__device__ __forceinline__ float bf16_to_f32(uint16_t b) {
    return __builtin_bit_cast(float, (uint32_t)b << 16);
}
// low / high half of a dword holding two bf16
__device__ __forceinline__ float bf16lo_to_f32(uint32_t w) {
    return __builtin_bit_cast(float, w << 16);
}
__device__ __forceinline__ float bf16hi_to_f32(uint32_t w) {
    return __builtin_bit_cast(float, w & 0xFFFF0000u);
}
// round-to-nearest-even fp32 -> bf16 (finite inputs)
__device__ __forceinline__ uint32_t f32_to_bf16_rne(float f) {
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return u >> 16;
}
// two fp32 -> one dword of two bf16 / two fp16, round to nearest even
// (v_cvt_pk_bf16_f32 / v_cvt_pk_f16_f32)
__device__ __forceinline__ uint32_t pack_bf16_rne(float lo, float hi) {
    typedef __attribute__((ext_vector_type(2))) float v2f;
    typedef __attribute__((ext_vector_type(2))) __bf16 v2b;
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f){lo, hi}, v2b));
}
__device__ __forceinline__ uint32_t pack_f16_rne(float lo, float hi) {
    typedef __attribute__((ext_vector_type(2))) float v2f;
    typedef __attribute__((ext_vector_type(2))) _Float16 v2h;
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f){lo, hi}, v2h));
}
// acc + both halves of a dword of two bf16 / two fp16, in fp32 (one dot-product instruction)
__device__ __forceinline__ float pair_sum_bf16(uint32_t w, float acc) {
    typedef __attribute__((ext_vector_type(2))) __bf16 v2b;
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2b, w), __builtin_bit_cast(v2b, 0x3F803F80u), acc, false);
}
__device__ __forceinline__ float pair_sum_f16(uint32_t w, float acc) {
    typedef __attribute__((ext_vector_type(2))) _Float16 v2h;
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(v2h, w), __builtin_bit_cast(v2h, 0x3C003C00u), acc, false);
}
// Two E4M3 bytes -> one dword of two fp16 (exact: E4M3 fits fp16's normal range)
template <bool HI>
__device__ __forceinline__ uint32_t e4m3x2_to_f16x2(uint32_t w) {
    typedef __attribute__((ext_vector_type(2))) _Float16 v2h;
    v2h r = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8((int)w, 1.0f, HI);
    return __builtin_bit_cast(uint32_t, r);
}
// Two E4M3 bytes (low or high 16 bits of w) -> two fp32, hardware conversion
// (OCP E4M3fn on gfx950).
template <bool HI>
__device__ __forceinline__ f32x2 e4m3x2_to_f32(uint32_t w) {
    return __builtin_amdgcn_cvt_pk_f32_fp8((int)w, HI);
}
// Two E4M3 bytes -> one dword of two bf16.  Every E4M3 value is exactly
// representable in bf16, so the conversion is exact.
template <bool HI>
__device__ __forceinline__ uint32_t e4m3x2_to_bf16x2(uint32_t w) {
    bf16x2 r = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)w, 1.0f, HI);
    return __builtin_bit_cast(uint32_t, r);
}

// what place N of this lane's row of sixteen lanes holds (DPP row broadcast)
template <int N>
__device__ __forceinline__ uint32_t row_place(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x150 + N, 0xF, 0xF, true);
}
// Lane l meets lane l ^ 16 (l ^ 32) without a trip through LDS: the rows of sixteen lanes (the
// halves of the wave) trade places between two copies of the value, and a commutative
// operation on the two copies is what a butterfly step would give, bit for bit.
__device__ __forceinline__ void lanes_swap16(uint32_t &a, uint32_t &b) {
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}
__device__ __forceinline__ void lanes_swap32(uint32_t &a, uint32_t &b) {
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}
// x / d for x < 2^25 and d <= 64, from 2^31 / d rounded up (a division is thirty instructions); with d up to
// 1024 and such x the quotient may be one too large
inline uint32_t div_inverse(uint32_t d) { return (uint32_t)((((uint64_t)1 << 31) + d - 1) / d); }
__device__ __forceinline__ uint32_t div_by(uint32_t x, uint32_t inv) { return (uint32_t)(((uint64_t)(2 * x) * inv) >> 32); }
// max(v[l], v[l ^ 16]) and max(v[l], v[l ^ 32]) in every lane
__device__ __forceinline__ uint32_t lanes_xor16_max(uint32_t v) {
    uint32_t a = v, b = v;
    lanes_swap16(a, b);
    return a > b ? a : b;
}
__device__ __forceinline__ uint32_t lanes_xor32_max(uint32_t v) {
    uint32_t a = v, b = v;
    lanes_swap32(a, b);
    return a > b ? a : b;
}
__device__ __forceinline__ float xor16_max(float v) {
    uint32_t a = __builtin_bit_cast(uint32_t, v), b = a;
    lanes_swap16(a, b);
    return fmaxf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
}
__device__ __forceinline__ float xor32_max(float v) {
    uint32_t a = __builtin_bit_cast(uint32_t, v), b = a;
    lanes_swap32(a, b);
    return fmaxf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
}
__device__ __forceinline__ float xor16_sum(float v) {
    uint32_t a = __builtin_bit_cast(uint32_t, v), b = a;
    lanes_swap16(a, b);
    return __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b);
}
__device__ __forceinline__ float xor32_sum(float v) {
    uint32_t a = __builtin_bit_cast(uint32_t, v), b = a;
    lanes_swap32(a, b);
    return __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b);
}
// Reductions and scans over the wave without LDS.  Within a row of sixteen lanes through DPP:
// swap in pairs, swap pairs, mirror the half row, mirror the row (every step joins two groups
// of lanes that already agree, so all lanes end with the result); across rows the two swaps
// above.  A scan shifts within the row by 1, 2, 4, 8 and then hands the last lane of a row to
// the rows behind it.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK, 0xF, false);   // lanes without a source read 0
}
#define CWICK_WAVE_ALLREDUCE(v, OP)                                                         \
    do {                                                                                    \
        { const uint32_t o_ = dpp_u32<0xB1, 0xF>(v); v = OP(v, o_); }   /* quad_perm [1,0,3,2] */ \
        { const uint32_t o_ = dpp_u32<0x4E, 0xF>(v); v = OP(v, o_); }   /* quad_perm [2,3,0,1] */ \
        { const uint32_t o_ = dpp_u32<0x141, 0xF>(v); v = OP(v, o_); }  /* row_half_mirror */      \
        { const uint32_t o_ = dpp_u32<0x140, 0xF>(v); v = OP(v, o_); }  /* row_mirror */           \
        { uint32_t a_ = v, b_ = v; lanes_swap16(a_, b_); v = OP(a_, b_); }                  \
        { uint32_t a_ = v, b_ = v; lanes_swap32(a_, b_); v = OP(a_, b_); }                  \
    } while (0)
#define CWICK_OP_ADD(a, b) ((a) + (b))
#define CWICK_OP_MAX(a, b) ((a) > (b) ? (a) : (b))
#define CWICK_OP_MIN(a, b) ((a) < (b) ? (a) : (b))
__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t v) { CWICK_WAVE_ALLREDUCE(v, CWICK_OP_ADD); return v; }
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) { CWICK_WAVE_ALLREDUCE(v, CWICK_OP_MAX); return v; }
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) { CWICK_WAVE_ALLREDUCE(v, CWICK_OP_MIN); return v; }
// inclusive prefix sum over the lanes of the wave
__device__ __forceinline__ uint32_t wave_scan_u32(uint32_t v) {
    v += dpp_u32<0x111, 0xF>(v);     // row_shr:1
    v += dpp_u32<0x112, 0xF>(v);     // row_shr:2
    v += dpp_u32<0x114, 0xF>(v);     // row_shr:4
    v += dpp_u32<0x118, 0xF>(v);     // row_shr:8
    v += dpp_u32<0x142, 0xA>(v);     // row_bcast:15 into rows 1 and 3
    v += dpp_u32<0x143, 0xC>(v);     // row_bcast:31 into rows 2 and 3
    return v;
}
// one step of a sum over aligned groups of lanes, every lane of the group ending with the total
// (a group of `width` lanes whose halves already hold their own totals): DPP inside a row of
// sixteen, the swaps across rows
template <int WIDTH>
__device__ __forceinline__ float group_step_sum(float v) {
    static_assert(WIDTH == 2 || WIDTH == 4 || WIDTH == 8 || WIDTH == 16 || WIDTH == 32 || WIDTH == 64, "group width");
    if (WIDTH == 32) return xor16_sum(v);
    if (WIDTH == 64) return xor32_sum(v);
    constexpr int CTRL = WIDTH == 2 ? 0xB1 : WIDTH == 4 ? 0x4E : WIDTH == 8 ? 0x141 : 0x140;
    return v + __builtin_bit_cast(float, dpp_u32<CTRL, 0xF>(__builtin_bit_cast(uint32_t, v)));
}
// the maximum over each row of sixteen lanes
__device__ __forceinline__ float row_max(float v) {
#define CWICK_ROW_MAX(ctrl)                                                                                   \
    v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xF, 0xF, false)))
    CWICK_ROW_MAX(0xB1);     // quad_perm [1, 0, 3, 2]
    CWICK_ROW_MAX(0x4E);     // quad_perm [2, 3, 0, 1]
    CWICK_ROW_MAX(0x141);    // row_half_mirror
    CWICK_ROW_MAX(0x140);    // row_mirror
#undef CWICK_ROW_MAX
    return v;
}
// the maximum over the wave in every lane
__device__ __forceinline__ float wave_max(float v) {
#define CWICK_DPP_MAX(ctrl)                                                                                   \
    v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xF, 0xF, false)))
    CWICK_DPP_MAX(0xB1);     // quad_perm [1, 0, 3, 2]
    CWICK_DPP_MAX(0x4E);     // quad_perm [2, 3, 0, 1]
    CWICK_DPP_MAX(0x141);    // row_half_mirror
    CWICK_DPP_MAX(0x140);    // row_mirror
#undef CWICK_DPP_MAX
    return xor32_max(xor16_max(v));
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// bf16 values of a query as two E4M3 terms, hi + lo, in units of a power of two that the lanes which hold the same
// head's block share.  The bf16 pairs go straight into the scaled conversions: nine instructions per pair, where widening,
// scaling and the plain conversions took thirteen (the same bits for every bf16 value below the unit's
// overflow).  The largest magnitude is an integer maximum of the bit patterns without their signs.
typedef __attribute__((ext_vector_type(2))) unsigned short q_u16x2;
__device__ __forceinline__ q_u16x2 q_larger(q_u16x2 m, uint32_t pair) {
    return __builtin_elementwise_max(m, __builtin_bit_cast(q_u16x2, pair & 0x7FFF7FFFu));
}
// the unit's E8M0 byte, from the largest magnitude's bits
__device__ __forceinline__ uint32_t q_unit(uint32_t top) {
    const int s = top ? (int)(top >> 7) - 127 - 7 : 0;
    return (uint32_t)(127 + (s < -110 ? -110 : s));
}
// four values, two pairs
__device__ __forceinline__ void q_two_terms(uint32_t x0, uint32_t x1, uint32_t unit_byte, uint32_t &hi, uint32_t &lo) {
    typedef __attribute__((ext_vector_type(2))) short s16x2;
    typedef __attribute__((ext_vector_type(2))) __bf16 b16x2;
    const float unit = __builtin_bit_cast(float, unit_byte << 23);
    s16x2 h = {0, 0}, l = {0, 0};
#define CWICK_Q_PAIR(x, HALF)                                                                                           \
    do {                                                                                                                \
        h = __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(h, __builtin_bit_cast(b16x2, x), unit, HALF);                     \
        const f32x2 back = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(__builtin_bit_cast(uint32_t, h), unit, HALF);       \
        l = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(l, bf16lo_to_f32(x) - back[0], bf16hi_to_f32(x) - back[1], unit, HALF); \
    } while (0)
    CWICK_Q_PAIR(x0, 0);
    CWICK_Q_PAIR(x1, 1);
#undef CWICK_Q_PAIR
    hi = __builtin_bit_cast(uint32_t, h);
    lo = __builtin_bit_cast(uint32_t, l);
}
// 32 values (16 dwords) per lane, the head's 128 dims in lanes l, l ^ 16, l ^ 32, l ^ 48; returns the unit's E8M0 byte
__device__ __forceinline__ uint32_t q_two_terms(const u32x4 (&w)[4], u32x4 (&hi)[2], u32x4 (&lo)[2]) {
    q_u16x2 m[4] = {};
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
        for (int d = 0; d < 4; d++) m[d] = q_larger(m[d], w[c][d]);
    const q_u16x2 mm = __builtin_elementwise_max(__builtin_elementwise_max(m[0], m[1]), __builtin_elementwise_max(m[2], m[3]));
    const uint32_t unit_byte = q_unit(lanes_xor32_max(lanes_xor16_max(mm[0] > mm[1] ? mm[0] : mm[1])));
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
        for (int d = 0; d < 4; d++) {
            uint32_t h, l;
            q_two_terms(w[2 * c + (d >> 1)][2 * (d & 1)], w[2 * c + (d >> 1)][2 * (d & 1) + 1], unit_byte, h, l);
            hi[c][d] = h;
            lo[c][d] = l;
        }
    return unit_byte;
}

// Sixteen bytes of host memory past every cache: plain accesses may find a line that an earlier kernel left
// in an L2, or leave one there until the kernel ends.
__device__ __forceinline__ u32x4 load_host16(const void *p) {
    const uint64_t a = __hip_atomic_load((const uint64_t *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    const uint64_t b = __hip_atomic_load((const uint64_t *)p + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return (u32x4){(uint32_t)a, (uint32_t)(a >> 32), (uint32_t)b, (uint32_t)(b >> 32)};
}
// Stores written through to memory as they are made: for the host, and for kernels that run on other XCDs
// (what sits dirty in an L2 is written back at the end of the kernel, on the critical path).  In assembly:
// as relaxed system-scope atomics the lanes' stores would leave one by one, a bus transaction each (16 KB
// to host memory took 130 us, 6 so).
__device__ __forceinline__ void store_through16(void *p, u32x4 v) {
    // (a store of more than 64 bits reads its data late: one wait state before the registers may be written)
    asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n\ts_nop 0" ::"v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ void store_through8(void *p, u32x2 v) {
    asm volatile("global_store_dwordx2 %0, %1, off sc0 sc1" ::"v"(p), "v"(v) : "memory");
}
// the wave's stores have been performed (those written through: where the host sees them)
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
__device__ __forceinline__ void host_flag(uint32_t *flags, int i, uint32_t epoch) {
    __hip_atomic_store(flags + i, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Round-to-nearest-even fp32 -> E4M3fn (the caller has clamped to +-448): the
// bit recipe of src/ds_quant.c:102-128, except that a round-up out of the last
// subnormal carries into the first normal (byte 0x08) instead of being masked
// away (`mm & 7u`, :127), so that the result is the nearest grid point as the
// reference's own round-trip check demands (tools/ds_verify.c:48-63).
__device__ __forceinline__ uint32_t f32_to_e4m3_rne(float v) {
    if (v == 0.0f) return 0u;
    uint32_t u = __builtin_bit_cast(uint32_t, v);
    uint32_t sign = u >> 31;
    int32_t exp = (int32_t)((u >> 23) & 0xFFu) - 127;
    uint32_t m24 = (1u << 23) | (u & 0x7FFFFFu);
    if (exp >= -6) {
        uint32_t keep = m24 >> 20;
        uint32_t rem = m24 & 0xFFFFFu;
        if (rem > 0x80000u || (rem == 0x80000u && (keep & 1u))) keep++;
        int32_t e = exp;
        if (keep == 16u) { keep >>= 1; e++; }
        if (e > 8) { keep = 14u; e = 8; }
        return (sign << 7) | ((uint32_t)(e + 7) << 3) | (keep & 7u);
    }
    if (exp < -10) return sign << 7;
    int32_t sh = 14 - exp;
    uint32_t mm = m24 >> sh;
    uint32_t rem = m24 & ((1u << sh) - 1u);
    uint32_t half = 1u << (sh - 1);
    if (rem > half || (rem == half && (mm & 1u))) mm++;
    return (sign << 7) | mm;
}

}  // namespace cwick
