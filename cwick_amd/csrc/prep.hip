// prep.hip -- the steps on either side of the attention kernels, kept on the device so that the
// queries and the outputs never cross the host link:
//
//   mla_absorb   q_abs[h] = W_k[h]^T q_nope[h]  (+ the rope dims of q passed through), narrowed to
//                the bf16 the MLA kernels take   (src/attention.c:741-744, gemv_bf16_t :145-177)
//   mla_expand   attn_out[h] = W_v[h] c_acc[h]    (src/attention.c:812-815, gemv_bf16_n :184-224)
//   gqa_prepare  per-head RMS norm with (1 + w) weights, partial rotate-half RoPE, Q narrowed to
//                bf16, K and V rows narrowed and appended to the device cache
//                (src/q35_model.c:1627-1652; rms_norm_w :111-121, rope_apply :144-153)
//
// All three are bandwidth-bound passes over small operands (the kv_b_proj slice of a layer is
// 128 heads x 320 rows x 512 bf16 = 42 MB; a decode step of the norm touches 20 heads).  The
// sums are fp32 like the reference's; their order is the wave's tree, not the CPU's serial
// loop, so results agree to rounding, not bit for bit.
#include "common.hpp"

#include <type_traits>

namespace cwick {
namespace {

// Absorb and expand stream one half of kv_b_proj (64 heads: 8.4 MB) past one or a few queries: what
// bounds them is how much of it is on its way at once.  A head is shared by four workgroups, so that
// 64 heads are 256 of them, and every thread requests its 128 bytes of the weights before it touches
// a query; the same registers then serve up to PROJ_QUERIES queries.  (One workgroup per head and
// query, eight rows on their way: 64 heads, one query 7.6 us for absorb and 19.2 us for expand.)
constexpr int PROJ_SPLIT = 4;            // workgroups per head
constexpr int PROJ_QUERIES = 4;          // queries per workgroup
constexpr int PROJ_ROWS = 8;             // 16-byte pieces of the weights per thread

// 16-byte loads that promise no more than dword alignment (what the entry points ask for)
typedef u32x4 __attribute__((aligned(4))) u32x4_a4;
typedef f32x4 __attribute__((aligned(4))) f32x4_a4;

// Sums over the lanes of pairs of values at a time: in each pair one of two lane groups gets the first value's
// sum and the other the second's, for one swap and one addition.
// x[i] and x[i + N / 2] -> x[i], lanes 0 .. 31 and 32 .. 63
template <int N>
__device__ __forceinline__ void halve32(float (&x)[N]) {
#pragma unroll
    for (int i = 0; i < N / 2; i++) {
        uint32_t a = __builtin_bit_cast(uint32_t, x[i]), b = __builtin_bit_cast(uint32_t, x[i + N / 2]);
        lanes_swap32(a, b);
        x[i] = __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b);
    }
}
// the same for the rows of sixteen lanes, even and odd
template <int N>
__device__ __forceinline__ void halve16(float (&x)[N], int n) {
#pragma unroll
    for (int i = 0; i < N / 2; i++)
        if (i < n / 2) {
            uint32_t a = __builtin_bit_cast(uint32_t, x[i]), b = __builtin_bit_cast(uint32_t, x[i + n / 2]);
            lanes_swap16(a, b);
            x[i] = __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b);
        }
}

// within the rows: the value of the lane opposite in a group of sixteen, eight (bit 3 or 2 of the lane differs, and
// the bits below it) or four lanes (bit 1 does)
template <int WIDTH>
__device__ __forceinline__ float opposite(float v) {
    constexpr int CTRL = WIDTH == 4 ? 0x4E : WIDTH == 8 ? 0x141 : 0x140;
    return __builtin_bit_cast(float, dpp_u32<CTRL, 0xF>(__builtin_bit_cast(uint32_t, v)));
}

// workgroup (4 head + block, NY queries): columns 128 block .. +128 of the 512-wide latent.  Sixteen
// lanes read a row's 256 bytes, so the 256 threads hold sixteen rows, PROJ_ROWS times; the sixteen
// partial sums of a column meet through lane swaps and, between the waves, in LDS.
// Bound by the weights for one query (8.4 MB at 64 heads: 3.8 us, 4.3 with the rope dims fetched at the end).  For more of them it is the instructions of the one
// or two waves that a SIMD has: so a weight is widened once for all NY queries, their values of a row are one read,
// and the swaps sum two values at a time.  (A query after the other, each with its own sums, and the rope dims
// fetched at the end: 7.6 us for four queries of 64 heads, 4.8 now; of 128 heads 9.4, 6.5.)
template <int NY>
__global__ void __launch_bounds__(256)
mla_absorb_kernel(const uint16_t *__restrict__ kvb_w, const float *__restrict__ q, int64_t q_stride, int batch,
                  int q_dim, int nope, int rope, int kv_dim, int kv_lora, uint16_t *__restrict__ out) {
    constexpr int COLS = CWICK_HIP_LATENT_VDIM / PROJ_SPLIT, ROWS = 16, STEP = ROWS * PROJ_ROWS;
    static_assert(COLS == 16 * 8, "sixteen lanes of eight columns");
    static_assert(STEP == 128 && CWICK_HIP_LATENT_KDIM - CWICK_HIP_LATENT_VDIM == 64 && NY <= 4, "rows and rope dims by the thread");
    typedef float vec __attribute__((ext_vector_type(NY)));
    const int h = blockIdx.x / PROJ_SPLIT, blk = blockIdx.x % PROJ_SPLIT, nh = gridDim.x / PROJ_SPLIT;
    const int y0 = blockIdx.y * PROJ_QUERIES, ny = batch - y0 < NY ? batch - y0 : NY;
    const int tid = threadIdx.x, c8 = tid & 15, rg = tid >> 4;
    __shared__ __attribute__((aligned(16))) float qs[512][NY];
    __shared__ __attribute__((aligned(16))) float part[NY][4][COLS];
    const uint16_t *wk = kvb_w + (size_t)h * kv_dim * kv_lora + blk * COLS + c8 * 8;
    u32x4 w[PROJ_ROWS];
#pragma unroll
    for (int j = 0; j < PROJ_ROWS; j++) {
        const int r = rg + ROWS * j;
        w[j] = *(const u32x4_a4 *)(wk + (size_t)(r < nope ? r : 0) * kv_lora);     // nope >= 1 (the launcher)
    }
    // the rope dims of the query pass through (zero when the model has none): wave y has query y's
    const float *qh = q + (size_t)y0 * q_stride + (size_t)h * q_dim;
    const int yr = tid >> 6, ir = tid & 63;
    float x_rope = 0.0f;
    if (blk == 0 && yr < ny && ir < rope) x_rope = qh[(size_t)yr * q_stride + nope + ir];
    // rows past `nope` and queries past the batch meet a zero
    for (int i = tid & 127; i < nope + STEP - 1; i += STEP)
#pragma unroll
        for (int k = 0; k < (NY + 1) / 2; k++) {
            const int y = (tid >> 7) + 2 * k;
            if (i < 512 && y < NY) qs[i][y] = i < nope && y < ny ? qh[(size_t)y * q_stride + i] : 0.0f;
        }
    __syncthreads();
    float a[NY * 8];                                                // [query][column]
#pragma unroll
    for (int i = 0; i < NY * 8; i++) a[i] = 0.0f;
    for (int r0 = 0; r0 < nope; r0 += STEP) {
        if (r0)
#pragma unroll
            for (int j = 0; j < PROJ_ROWS; j++) {
                const int r = r0 + rg + ROWS * j;
                w[j] = *(const u32x4_a4 *)(wk + (size_t)(r < nope ? r : 0) * kv_lora);
            }
#pragma unroll
        for (int j = 0; j < PROJ_ROWS; j++) {
            const vec x = *(const vec *)qs[r0 + rg + ROWS * j];
#pragma unroll
            for (int d = 0; d < 4; d++) {
                const float lo = bf16lo_to_f32(w[j][d]), hi = bf16hi_to_f32(w[j][d]);
#pragma unroll
                for (int y = 0; y < NY; y++) {
                    a[8 * y + 2 * d] = __builtin_fmaf(x[y], lo, a[8 * y + 2 * d]);
                    a[8 * y + 2 * d + 1] = __builtin_fmaf(x[y], hi, a[8 * y + 2 * d + 1]);
                }
            }
        }
    }
    // row g of sixteen lanes ends with the eight columns of query g (of two queries: g / 2, of one: every row)
    if (NY > 1) halve32(a);
    if (NY > 2) halve16(a, NY * 4);
#pragma unroll
    for (int d = 0; d < 8; d++) {
        if (NY == 1) a[d] = xor32_sum(a[d]);
        if (NY <= 2) a[d] = xor16_sum(a[d]);
    }
    const int g = (tid & 63) >> 4;
    if (NY == 4 || (g & (NY == 2 ? 1 : 3)) == 0) {
        float *dst = &part[NY == 4 ? g : NY == 2 ? g >> 1 : 0][tid >> 6][c8 * 8];
        *(f32x4 *)dst = (f32x4){a[0], a[1], a[2], a[3]};
        *(f32x4 *)(dst + 4) = (f32x4){a[4], a[5], a[6], a[7]};
    }
    __syncthreads();
    uint16_t *o = out + ((size_t)y0 * nh + h) * CWICK_HIP_LATENT_KDIM;
    const size_t o_query = (size_t)nh * CWICK_HIP_LATENT_KDIM;
    for (int i = tid; i < ny * COLS / 2; i += 256) {
        const int y = i / (COLS / 2), c = i % (COLS / 2) * 2;
        f32x2 t = *(const f32x2 *)&part[y][0][c];
#pragma unroll
        for (int v = 1; v < 4; v++) {
            const f32x2 x = *(const f32x2 *)&part[y][v][c];
            t[0] += x[0], t[1] += x[1];
        }
        *(uint32_t *)(o + y * o_query + blk * COLS + c) = pack_bf16_rne(t[0], t[1]);
    }
    if (blk == 0 && yr < ny) o[yr * o_query + kv_lora + ir] = (uint16_t)f32_to_bf16_rne(x_rope);
}

// workgroup (4 head + block, NY queries): the rows of W_v with (row / 8) % 16 = 4 block + wave.  A lane
// reads eight bf16 of a row (16 bytes, a wave the row's KiB) and keeps the matching eight floats of the
// queries' c_acc; the 8 NY dots of a wave are summed over the lanes two at a time, so that every lane ends with one.
// (Each query by itself, its sums in all lanes: 6.0 us for four queries of 64 heads, 3.9 now; one query 3.8, 3.4.)
template <int NY>
__global__ void __launch_bounds__(256)
mla_expand_kernel(const uint16_t *__restrict__ kvb_w, const float *__restrict__ c_acc, int batch, int nope, int vdim,
                  int kv_dim, int kv_lora, float *__restrict__ out) {
    static_assert(CWICK_HIP_LATENT_VDIM == 64 * 8 && PROJ_ROWS == 8, "a wave's lanes cover a row");
    const int h = blockIdx.x / PROJ_SPLIT, blk = blockIdx.x % PROJ_SPLIT, nh = gridDim.x / PROJ_SPLIT;
    const int y0 = blockIdx.y * PROJ_QUERIES, ny = batch - y0 < NY ? batch - y0 : NY;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint16_t *wv = kvb_w + ((size_t)h * kv_dim + nope) * kv_lora + 8 * lane;
    f32x4 c[NY][2];
#pragma unroll
    for (int y = 0; y < NY; y++) {
        const float *p = c_acc + ((size_t)(y0 + (y < ny ? y : 0)) * nh + h) * kv_lora + 8 * lane;
        c[y][0] = *(const f32x4_a4 *)p, c[y][1] = *(const f32x4_a4 *)(p + 4);
    }
    for (int r0 = (blk * 4 + wave) * PROJ_ROWS; r0 < vdim; r0 += PROJ_SPLIT * 4 * PROJ_ROWS) {
        u32x4 w[PROJ_ROWS];
#pragma unroll
        for (int j = 0; j < PROJ_ROWS; j++)
            w[j] = *(const u32x4_a4 *)(wv + (size_t)(r0 + j < vdim ? r0 + j : 0) * kv_lora);
        float s[NY * 8];                                            // [query][row]
#pragma unroll
        for (int j = 0; j < PROJ_ROWS; j++) {
            float e[8];
#pragma unroll
            for (int d = 0; d < 4; d++) e[2 * d] = bf16lo_to_f32(w[j][d]), e[2 * d + 1] = bf16hi_to_f32(w[j][d]);
#pragma unroll
            for (int y = 0; y < NY; y++) {
                float t = e[0] * c[y][0][0];
#pragma unroll
                for (int d = 1; d < 8; d++) t = __builtin_fmaf(e[d], c[y][d >> 2][d & 3], t);
                s[8 * y + j] = t;
            }
        }
        // Lane bits 5, 4, 3, 2, 1 (as many as there are halvings) pick the value that the lane ends with, the first one
        // the upper half of the list; what is left of the lanes adds up the same value.
        halve32(s);
        halve16(s, NY * 4);
        constexpr int LEFT = NY * 2;                                // values a lane has now
        auto halve = [&](auto width, int n) {
            constexpr int W = decltype(width)::value;
            const bool upper = lane & (W / 2);                      // (the lanes of a group that differ in lower bits hold the same values)
#pragma unroll
            for (int i = 0; i < LEFT / 2; i++)
                if (i < n / 2) {
                    const float keep = upper ? s[i + n / 2] : s[i], give = upper ? s[i] : s[i + n / 2];
                    s[i] = keep + opposite<W>(give);
                }
        };
        if (LEFT == 8) halve(std::integral_constant<int, 16>{}, 8);
        if (LEFT >= 4) halve(std::integral_constant<int, LEFT == 8 ? 8 : 16>{}, 4);
        halve(std::integral_constant<int, LEFT == 8 ? 4 : LEFT == 4 ? 8 : 16>{}, 2);
        float t = s[0];
        if (LEFT <= 2) t = group_step_sum<8>(group_step_sum<4>(group_step_sum<2>(t)));
        else if (LEFT == 4) t = group_step_sum<4>(group_step_sum<2>(t));
        else t = group_step_sum<2>(t);
        const int bits = NY == 4 ? lane >> 1 : NY == 2 ? lane >> 2 : lane >> 3, y = bits >> 3, j = bits & 7;
        const bool first = (lane & (NY == 4 ? 1 : NY == 2 ? 3 : 7)) == 0;
        if (first && y < ny && r0 + j < vdim) out[((size_t)(y0 + y) * nh + h) * vdim + r0 + j] = t;
    }
}

// one wave per (token, head), q heads first, then k heads, then v heads (narrowed only)
//
// Bound by memory (517 positions of 16 + 2 x 4 heads read 12.7 MB and write 6.4), which takes all of a
// head's operands on their way at once: a lane holds four neighbouring dims, asks for its rotation
// partner's values and weights next to its own, and nothing goes through LDS.  (One dim per lane and
// load, the partner through LDS, the head found by a 64-bit division: see gqa_prepare_kernel, which is
// left with the rotations whose halves are not in fours; 10 us for those 517 positions, 8.5 here.)
__global__ void __launch_bounds__(256)
gqa_prepare4_kernel(const float *__restrict__ q_proj, int64_t q_head_stride, const float *__restrict__ k_proj,
                    const float *__restrict__ v_proj, int64_t pos0, int H, int KV, int HD,
                    const float *__restrict__ q_norm, const float *__restrict__ k_norm, float eps,
                    const float *__restrict__ rope_cos, const float *__restrict__ rope_sin, int rotary,
                    uint16_t *__restrict__ q_out, uint16_t *__restrict__ k_cache, uint16_t *__restrict__ v_cache) {
    const int d = (threadIdx.x & 63) * 4;
    const int hh = blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (hh >= H + 2 * KV) return;
    const size_t t = blockIdx.x, p = (size_t)pos0 + t;
    const float *src, *w = nullptr;
    uint16_t *dst;
    if (hh < H) {
        src = q_proj + (t * H + hh) * q_head_stride;
        w = q_norm;
        dst = q_out + (t * H + hh) * HD;
    } else if (hh < H + KV) {
        src = k_proj + (t * KV + (hh - H)) * HD;
        w = k_norm;
        dst = k_cache + (p * KV + (hh - H)) * HD;
    } else {
        src = v_proj + (t * KV + (hh - H - KV)) * HD;
        dst = v_cache + (p * KV + (hh - H - KV)) * HD;
    }
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f}, one = {1.0f, 1.0f, 1.0f, 1.0f};
    f32x4 v = d < HD ? *(const f32x4_a4 *)(src + d) : zero;
    if (hh < H + KV) {
        const int pairs = rotary / 2;
        const bool turns = d < rotary, first = d < pairs;
        const int mate = first ? d + pairs : d - pairs;
        f32x4 g = one, x = zero, gx = one, cs = one, sn = zero;
        if (turns) {
            x = *(const f32x4_a4 *)(src + mate);
            cs = *(const f32x4_a4 *)(rope_cos + p * pairs + (first ? d : mate));
            sn = *(const f32x4_a4 *)(rope_sin + p * pairs + (first ? d : mate));
        }
        if (w) {
            if (d < HD) g = one + *(const f32x4_a4 *)(w + d);
            if (turns) gx = one + *(const f32x4_a4 *)(w + mate);
        }
        float acc = v[0] * v[0];
#pragma unroll
        for (int i = 1; i < 4; i++) acc = __builtin_fmaf(v[i], v[i], acc);
        acc = wave_sum(acc);
        const float rstd = 1.0f / sqrtf(acc / (float)HD + eps);
        const float sign = first ? -1.0f : 1.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            v[i] = v[i] * rstd * g[i];
            if (turns) v[i] = v[i] * cs[i] + sign * (x[i] * rstd * gx[i] * sn[i]);
        }
    }
    if (d < HD) *(u32x2 *)(dst + d) = (u32x2){pack_bf16_rne(v[0], v[1]), pack_bf16_rne(v[2], v[3])};
}

// the same for any rotation
__global__ void __launch_bounds__(256)
gqa_prepare_kernel(const float *__restrict__ q_proj, int64_t q_head_stride, const float *__restrict__ k_proj,
                   const float *__restrict__ v_proj, int64_t n, int64_t pos0, int H, int KV, int HD,
                   const float *__restrict__ q_norm, const float *__restrict__ k_norm, float eps,
                   const float *__restrict__ rope_cos, const float *__restrict__ rope_sin, int rotary,
                   uint16_t *__restrict__ q_out, uint16_t *__restrict__ k_cache, uint16_t *__restrict__ v_cache) {
    __shared__ float buf[4][256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int per_tok = H + 2 * KV;
    const int64_t item = (int64_t)blockIdx.x * 4 + wave;
    if (item >= n * per_tok) return;
    const int64_t t = item / per_tok;
    const int hh = (int)(item % per_tok);
    const int64_t p = pos0 + t;
    const float *src;
    const float *w = nullptr;
    uint16_t *dst;
    bool rot = true;
    if (hh < H) {
        src = q_proj + ((size_t)t * H + hh) * q_head_stride;
        w = q_norm;
        dst = q_out + ((size_t)t * H + hh) * HD;
    } else if (hh < H + KV) {
        src = k_proj + ((size_t)t * KV + (hh - H)) * HD;
        w = k_norm;
        dst = k_cache + ((size_t)p * KV + (hh - H)) * HD;
    } else {
        src = v_proj + ((size_t)t * KV + (hh - H - KV)) * HD;
        dst = v_cache + ((size_t)p * KV + (hh - H - KV)) * HD;
        rot = false;
    }
    float v[4];
    float acc = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int d = lane + 64 * i;
        v[i] = d < HD ? src[d] : 0.0f;
        acc = __builtin_fmaf(v[i], v[i], acc);
    }
    if (rot) {
        acc = wave_sum(acc);
        const float rstd = 1.0f / sqrtf(acc / (float)HD + eps);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int d = lane + 64 * i;
            if (d < HD) {
                const float x = v[i] * rstd;
                buf[wave][d] = w ? x * (1.0f + w[d]) : x;
            }
        }
        // the partner element of the rotation was written by another lane of this wave: LDS
        // serves a wave's instructions in order, the barrier only pins the compiler's order
        __builtin_amdgcn_wave_barrier();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        const int pairs = rotary / 2;
        const float *cs = rope_cos + (size_t)p * pairs, *sn = rope_sin + (size_t)p * pairs;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int d = lane + 64 * i;
            if (d >= HD) continue;
            float x = buf[wave][d];
            if (d < pairs) {
                const float b = buf[wave][d + pairs];
                x = x * cs[d] - b * sn[d];
            } else if (d < 2 * pairs) {
                const float a = buf[wave][d - pairs];
                x = x * cs[d - pairs] + a * sn[d - pairs];
            }
            v[i] = x;
        }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int d = lane + 64 * i;
        if (d < HD) dst[d] = (uint16_t)f32_to_bf16_rne(v[i]);
    }
}

}  // namespace

int launch_mla_absorb(const uint16_t *kvb_w, const float *q, int64_t q_stride, int batch, int n_heads,
                      int q_dim, int nope, int rope, int kv_dim, int kv_lora, uint16_t *q_abs, hipStream_t s) {
    CWICK_REQUIRE(kvb_w && q && q_abs, "mla_absorb: null pointer");
    CWICK_REQUIRE(batch >= 1 && batch <= 65535 && n_heads >= 1 && n_heads <= 65535, "mla_absorb: batch %d, n_heads %d",
                  batch, n_heads);
    CWICK_REQUIRE(kv_lora == CWICK_HIP_LATENT_VDIM, "mla_absorb: kv_lora %d (the latent cache holds 512)", kv_lora);
    CWICK_REQUIRE(nope >= 1 && rope >= 0 && rope <= CWICK_HIP_LATENT_KDIM - CWICK_HIP_LATENT_VDIM && nope + rope <= q_dim &&
                      nope + rope <= 512 && nope <= kv_dim,
                  "mla_absorb: nope %d rope %d q_dim %d kv_dim %d", nope, rope, q_dim, kv_dim);
    CWICK_REQUIRE((uintptr_t)kvb_w % 4 == 0 && (uintptr_t)q_abs % 4 == 0, "mla_absorb: operands must be 4-byte aligned");
    (batch == 1 ? mla_absorb_kernel<1> : batch == 2 ? mla_absorb_kernel<2> : mla_absorb_kernel<PROJ_QUERIES>)<<<
        dim3(n_heads * PROJ_SPLIT, (batch + PROJ_QUERIES - 1) / PROJ_QUERIES), 256, 0, s>>>(
        kvb_w, q, q_stride, batch, q_dim, nope, rope, kv_dim, kv_lora, q_abs);
    CWICK_HIP_CALL(hipGetLastError());
    return 1;
}

int launch_mla_expand(const uint16_t *kvb_w, const float *c_acc, int batch, int n_heads, int nope, int vdim,
                      int kv_dim, int kv_lora, float *out, hipStream_t s) {
    CWICK_REQUIRE(kvb_w && c_acc && out, "mla_expand: null pointer");
    CWICK_REQUIRE(batch >= 1 && batch <= 65535 && n_heads >= 1 && n_heads <= 65535, "mla_expand: batch %d, n_heads %d",
                  batch, n_heads);
    CWICK_REQUIRE(kv_lora == CWICK_HIP_LATENT_VDIM, "mla_expand: kv_lora %d (the latent cache holds 512)", kv_lora);
    CWICK_REQUIRE(vdim >= 1 && nope >= 0 && nope + vdim <= kv_dim, "mla_expand: nope %d vdim %d kv_dim %d", nope, vdim, kv_dim);
    CWICK_REQUIRE((uintptr_t)kvb_w % 16 == 0, "mla_expand: kv_b_proj must be 16-byte aligned");
    (batch == 1 ? mla_expand_kernel<1> : batch == 2 ? mla_expand_kernel<2> : mla_expand_kernel<PROJ_QUERIES>)<<<
        dim3(n_heads * PROJ_SPLIT, (batch + PROJ_QUERIES - 1) / PROJ_QUERIES), 256, 0, s>>>(
        kvb_w, c_acc, batch, nope, vdim, kv_dim, kv_lora, out);
    CWICK_HIP_CALL(hipGetLastError());
    return 1;
}

int launch_gqa_prepare(const float *q_proj, int64_t q_head_stride, const float *k_proj, const float *v_proj,
                       int64_t n, int64_t pos0, int n_heads, int n_kv_heads, int head_dim, const float *q_norm,
                       const float *k_norm, float eps, const float *rope_cos, const float *rope_sin, int rotary_dim,
                       uint16_t *q_out, uint16_t *k_cache, uint16_t *v_cache, hipStream_t s) {
    CWICK_REQUIRE(q_proj && k_proj && v_proj && q_out && k_cache && v_cache, "gqa_prepare: null pointer");
    CWICK_REQUIRE(n >= 1 && pos0 >= 0 && n <= ((int64_t)1 << 24), "gqa_prepare: n %lld pos0 %lld", (long long)n, (long long)pos0);
    CWICK_REQUIRE(head_dim >= 2 && head_dim <= 256, "gqa_prepare: head_dim %d (at most 256)", head_dim);
    CWICK_REQUIRE(n_heads >= 1 && n_kv_heads >= 1 && q_head_stride >= head_dim, "gqa_prepare: heads %d/%d, stride %lld",
                  n_heads, n_kv_heads, (long long)q_head_stride);
    CWICK_REQUIRE(rotary_dim >= 0 && rotary_dim <= head_dim && rotary_dim % 2 == 0, "gqa_prepare: rotary_dim %d", rotary_dim);
    CWICK_REQUIRE(rotary_dim == 0 || (rope_cos && rope_sin), "gqa_prepare: rope tables missing");
    // a rotation whose halves are in fours (every source is read in fours at dword alignment)
    if (head_dim % 4 == 0 && rotary_dim % 8 == 0 && (int64_t)n_heads + 2 * (int64_t)n_kv_heads <= 4 * 65535 &&
        ((uintptr_t)q_out | (uintptr_t)k_cache | (uintptr_t)v_cache) % 8 == 0) {
        gqa_prepare4_kernel<<<dim3((unsigned)n, (unsigned)((n_heads + 2 * n_kv_heads + 3) / 4)), 256, 0, s>>>(
            q_proj, q_head_stride, k_proj, v_proj, pos0, n_heads, n_kv_heads, head_dim, q_norm, k_norm, eps, rope_cos, rope_sin,
            rotary_dim, q_out, k_cache, v_cache);
        CWICK_HIP_CALL(hipGetLastError());
        return 1;
    }
    const int64_t items = n * (n_heads + 2 * n_kv_heads);
    gqa_prepare_kernel<<<dim3((unsigned)((items + 3) / 4)), 256, 0, s>>>(
        q_proj, q_head_stride, k_proj, v_proj, n, pos0, n_heads, n_kv_heads, head_dim, q_norm, k_norm, eps, rope_cos,
        rope_sin, rotary_dim, q_out, k_cache, v_cache);
    CWICK_HIP_CALL(hipGetLastError());
    return 1;
}

}  // namespace cwick

// ---------------------------------------------------------------------------
// indexer key production, candidate blocks, dequantised read-back
// ---------------------------------------------------------------------------
namespace cwick {
namespace {

// One wave per closed pool (src/attention.c:486-525): layer-norm statistics of each of the kp
// raw key rows, a softmax over the pool slots of gate + position bias per dimension, the affine
// k_norm on the normalised rows, the weighted mean as the pool's key; then the row is quantised
// like every indexer key (one fp32 scale per row, amax / 448).  hd = 128: two dims per lane.
__global__ void __launch_bounds__(256)
ikeys_pool_kernel(const float *__restrict__ tail_k, const float *__restrict__ tail_g, const uint16_t *__restrict__ ape,
                  const float *__restrict__ knw, const float *__restrict__ knb, float eps, int kp, int64_t n_pools,
                  uint8_t *__restrict__ out_rows, float *__restrict__ out_scales, float *__restrict__ out_f32) {
    constexpr int HD = CWICK_HIP_INDEX_DIM;
    const int lane = threadIdx.x & 63;
    const int64_t pool = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (pool >= n_pools) return;
    const float *k = tail_k + (size_t)pool * kp * HD, *gt = tail_g + (size_t)pool * kp * HD;
    // statistics in double like the reference's (sums of 128 floats are exact there in all but
    // contrived rows, so the order of the wave reduction does not show)
    float mean[8], inv[8], kv[8][2];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        mean[i] = inv[i] = kv[i][0] = kv[i][1] = 0.0f;
        if (i < kp) {
            kv[i][0] = k[i * HD + lane];
            kv[i][1] = k[i * HD + 64 + lane];
            mean[i] = (float)(wave_sum((double)kv[i][0] + (double)kv[i][1]) / (double)HD);
            const double t0 = (double)kv[i][0] - (double)mean[i], t1 = (double)kv[i][1] - (double)mean[i];
            inv[i] = 1.0f / sqrtf((float)(wave_sum(t0 * t0 + t1 * t1) / (double)HD) + eps);
        }
    }
    float res[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int d = lane + 64 * h;
        float lg[8], mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            lg[i] = -INFINITY;
            if (i < kp) {
                lg[i] = gt[i * HD + d] + bf16_to_f32(ape[i * HD + d]);
                mx = lg[i] > mx ? lg[i] : mx;
            }
        }
        float den = 0.0f, acc = 0.0f;
        const float w = knw[d], bb = knb[d];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            if (i < kp) {
                const float p = expf(lg[i] - mx);
                den += p;
                const float nv = ((kv[i][h] - mean[i]) * inv[i]) * w + bb;
                acc += p * nv;
            }
        }
        res[h] = den > 0.0f ? acc / den : 0.0f;
    }
    if (out_f32) {
        out_f32[(size_t)pool * HD + lane] = res[0];
        out_f32[(size_t)pool * HD + 64 + lane] = res[1];
    }
    const float amax = wave_max(fmaxf(fabsf(res[0]), fabsf(res[1])));
    const float s = amax > 0.0f ? amax / 448.0f : 1.0f;
    if (lane == 0) out_scales[pool] = s;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        float v = res[h] / s;
        v = fminf(fmaxf(v, -448.0f), 448.0f);
        out_rows[(size_t)pool * HD + lane + 64 * h] = (uint8_t)f32_to_e4m3_rne(v);
    }
}

// block maxima of the scores, the partly filled last block forced in (src/ds_model.c:1127-1135)
__global__ void __launch_bounds__(256)
cand_blockmax_kernel(const float *__restrict__ scores, int64_t n, int bs, int64_t nblk, float *__restrict__ bsc) {
    const int lane = threadIdx.x & 63;
    const int64_t b = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int row = blockIdx.y;
    if (b >= nblk) return;
    const float *s = scores + (size_t)row * n;
    const int64_t lo = b * bs, hi = lo + bs < n ? lo + bs : n;
    float mx = -INFINITY;
    for (int64_t t = lo + lane; t < hi; t += 64) mx = s[t] > mx ? s[t] : mx;
    mx = wave_max(mx);
    if (lane == 0) bsc[(size_t)row * nblk + b] = b == nblk - 1 ? INFINITY : mx;
}

__global__ void __launch_bounds__(256)
cand_mark_kernel(const int32_t *__restrict__ blk, int64_t k, int64_t n, int bs, uint8_t *__restrict__ cand) {
    const int row = blockIdx.y;
    const int64_t i = (int64_t)blockIdx.x;                 // one workgroup per chosen block
    if (i >= k) return;
    const int32_t b = blk[(size_t)row * k + i];
    if (b < 0) return;
    const int64_t lo = (int64_t)b * bs, hi = lo + bs < n ? lo + bs : n;
    for (int64_t t = lo + threadIdx.x; t < hi; t += 256) cand[(size_t)row * n + t] = 1;
}

__global__ void __launch_bounds__(256) cand_clear_kernel(uint8_t *__restrict__ cand, int64_t total) {
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (; i < total; i += stride) cand[i] = 0;
}

// positions outside the candidate blocks cannot be selected (src/ds_model.c:1144-1147)
__global__ void __launch_bounds__(256)
cand_apply_kernel(float *__restrict__ scores, const uint8_t *__restrict__ cand, int64_t total) {
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (; i < total; i += stride)
        if (!cand[i]) scores[i] = -INFINITY;
}

template <int DIM, int BLOCK>
__global__ void __launch_bounds__(256)
dequant_rows_kernel(const uint8_t *__restrict__ rows, const float *__restrict__ scales, int64_t n, float *__restrict__ out) {
    constexpr int NBLK = (DIM + BLOCK - 1) / BLOCK;
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * 256, total = n * DIM;
    for (; i < total; i += stride) {
        const int64_t r = i / DIM;
        const int d = (int)(i % DIM);
        out[i] = e4m3x2_to_f32<false>((uint32_t)rows[i])[0] * scales[r * NBLK + d / BLOCK];
    }
}

}  // namespace

int launch_ikeys_pool(const float *tail_k, const float *tail_g, const uint16_t *ape, const float *knw, const float *knb,
                      float eps, int kpool, int64_t n_pools, uint8_t *out_rows, float *out_scales, float *out_f32,
                      hipStream_t s) {
    CWICK_REQUIRE(tail_k && tail_g && ape && knw && knb && out_rows && out_scales, "ikeys_pool: null pointer");
    CWICK_REQUIRE(kpool >= 1 && kpool <= 8, "ikeys_pool: kpool %d (1..8, src/attention.c:492)", kpool);
    CWICK_REQUIRE(n_pools >= 1 && n_pools <= ((int64_t)1 << 30), "ikeys_pool: n_pools %lld", (long long)n_pools);
    ikeys_pool_kernel<<<dim3((unsigned)((n_pools + 3) / 4)), 256, 0, s>>>(tail_k, tail_g, ape, knw, knb, eps, kpool,
                                                                        n_pools, out_rows, out_scales, out_f32);
    CWICK_HIP_CALL(hipGetLastError());
    return 1;
}

int launch_candidate_select(const float *scores, int batch, int64_t n, int block, int64_t topk_blocks, uint8_t *cand,
                            hipStream_t s) {
    CWICK_REQUIRE(scores && cand, "candidate_select: null pointer");
    CWICK_REQUIRE(batch >= 1 && batch <= 65535 && n >= 1 && n <= ((int64_t)1 << 30), "candidate_select: batch %d n %lld",
                  batch, (long long)n);
    CWICK_REQUIRE(block >= 1 && topk_blocks >= 1 && topk_blocks <= 65536, "candidate_select: block %d, blocks kept %lld",
                  block, (long long)topk_blocks);
    const int64_t nblk = (n + block - 1) / block;
    // (the top-k below keeps its own workspace slot, so the block scores can sit in this call's)
    CWICK_REQUIRE(nblk < 16384, "candidate_select: %lld blocks (at most 16383)", (long long)nblk);
    const size_t bsc_b = ((size_t)batch * nblk * 4 + 255) & ~(size_t)255;
    char *ws = (char *)workspace(s, bsc_b + (size_t)batch * topk_blocks * 4);
    if (!ws) return 0;                      // workspace() has recorded why
    float *bsc = (float *)ws;
    int32_t *blk = (int32_t *)(ws + bsc_b);
    cand_blockmax_kernel<<<dim3((unsigned)((nblk + 3) / 4), batch), 256, 0, s>>>(scores, n, block, nblk, bsc);
    CWICK_HIP_CALL(hipGetLastError());
    {
        const int64_t total = (int64_t)batch * n;
        int64_t blocks = (total + 255) / 256;
        if (blocks > 8192) blocks = 8192;
        cand_clear_kernel<<<dim3((unsigned)blocks), 256, 0, s>>>(cand, total);      // a kernel, not a memset: safe under graph capture
    }
    if (!launch_topk(bsc, batch, nblk, topk_blocks, blk, s)) return 0;
    cand_mark_kernel<<<dim3((unsigned)topk_blocks, batch), 256, 0, s>>>(blk, topk_blocks, n, block, cand);
    CWICK_HIP_CALL(hipGetLastError());
    return 1;
}

// The rest of indexer_select behind the pool scores (src/attention.c:585-620), one workgroup per
// query.  pools[want] are the chosen pools in ascending order (the top-k select's output);
// the list keeps the reference's order: the pools that score above the lowest chosen score in
// ascending order, then the pools that equal it, each as its kp positions c kp + r; the
// positions behind the last closed pool; then the query's own position unless `strict` or it is
// the last entry already (the reference tests sel[n-1] only, :618).  mode_whole: no more pools
// than wanted -- the list is the whole prefix 0 .. npos-1 and n_sel is -1 (:558-559).
// Entries behind the list are -1, which the attention kernels skip.
constexpr int GLM_THREADS = 256;
__global__ void __launch_bounds__(GLM_THREADS)
glm_expand_kernel(const float *__restrict__ scores, const int32_t *__restrict__ pools, int64_t want, int64_t n_comp,
                  int64_t npos, int kp, int strict, int mode_whole, int32_t *__restrict__ sel, int64_t max_sel,
                  int32_t *__restrict__ n_sel) {
    __shared__ uint32_t red[GLM_THREADS / 64];
    __shared__ uint32_t wave_gt[GLM_THREADS / 64], wave_eq[GLM_THREADS / 64];
    const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int32_t *out = sel + (size_t)row * max_sel;
    if (mode_whole) {
        for (int64_t i = tid; i < max_sel; i += GLM_THREADS) out[i] = i < npos ? (int32_t)i : -1;
        if (tid == 0 && n_sel) n_sel[row] = -1;
        return;
    }
    const float *sc = scores + (size_t)row * n_comp;
    const int32_t *pl = pools + (size_t)row * want;
    // the lowest chosen score, as the select's own order key (so that -0.0 == +0.0)
    uint32_t kmin = 0xFFFFFFFFu;
    for (int64_t i = tid; i < want; i += GLM_THREADS) {
        const int32_t c = pl[i];
        if (c >= 0) {
            const uint32_t k = topk_key(sc[c]);
            kmin = k < kmin ? k : kmin;
        }
    }
    kmin = wave_min_u32(kmin);
    if (lane == 0) red[wave] = kmin;
    __syncthreads();
    kmin = red[0];
#pragma unroll
    for (int w = 1; w < GLM_THREADS / 64; w++) kmin = red[w] < kmin ? red[w] : kmin;
    // how many chosen pools score above it (they come first), and the last pool at it (the list's
    // last pool entry)
    uint32_t n_gt = 0, eq_last = 0;                 // eq_last: pool index + 1
    for (int64_t i = tid; i < want; i += GLM_THREADS) {
        const int32_t c = pl[i];
        if (c < 0) continue;
        if (topk_key(sc[c]) > kmin) n_gt++;
        else eq_last = (uint32_t)c + 1u > eq_last ? (uint32_t)c + 1u : eq_last;
    }
    n_gt = wave_sum_u32(n_gt);
    eq_last = wave_max_u32(eq_last);
    __syncthreads();
    if (lane == 0) red[wave] = n_gt, wave_eq[wave] = eq_last;
    __syncthreads();
    n_gt = 0, eq_last = 0;
#pragma unroll
    for (int w = 0; w < GLM_THREADS / 64; w++) {
        n_gt += red[w];
        eq_last = wave_eq[w] > eq_last ? wave_eq[w] : eq_last;
    }
    // places: a running count of both kinds over chunks of the pool list
    uint32_t base_gt = 0, base_eq = 0;
    for (int64_t i0 = 0; i0 < want; i0 += GLM_THREADS) {
        const int64_t i = i0 + tid;
        const int32_t c = i < want ? pl[i] : -1;
        const bool gt = c >= 0 && topk_key(sc[c]) > kmin, eq = c >= 0 && !gt;
        const uint32_t sg = wave_scan_u32(gt ? 1u : 0u), se = wave_scan_u32(eq ? 1u : 0u);
        __syncthreads();
        if (lane == 63) wave_gt[wave] = sg, wave_eq[wave] = se;
        __syncthreads();
        uint32_t og = base_gt, oe = base_eq, tg = 0, te = 0;
#pragma unroll
        for (int w = 0; w < GLM_THREADS / 64; w++) {
            if (w < wave) og += wave_gt[w], oe += wave_eq[w];
            tg += wave_gt[w], te += wave_eq[w];
        }
        if (c >= 0) {
            const uint32_t place = gt ? og + sg - 1u : n_gt + oe + se - 1u;
            for (int r = 0; r < kp; r++) out[(size_t)place * kp + r] = c * kp + r;
        }
        base_gt += tg, base_eq += te;
    }
    __syncthreads();
    // the tail, the query itself, the padding: one thread (a handful of entries) and then all
    const int64_t n_pool = (int64_t)(base_gt + base_eq) * kp;
    const int64_t tail = npos % kp;
    int64_t n = n_pool + tail;
    for (int64_t r = tid; r < tail; r += GLM_THREADS) out[n_pool + r] = (int32_t)(npos - tail + r);
    // the list's last entry before the self rule: the tail's, else the last pool at the lowest score
    const int64_t last = tail > 0 ? npos - 1 : (eq_last ? (int64_t)(eq_last - 1u) * kp + kp - 1 : -1);
    const bool add_self = !strict && last != npos - 1;
    if (tid == 0 && add_self) out[n] = (int32_t)(npos - 1);
    if (add_self) n++;
    for (int64_t i = n + tid; i < max_sel; i += GLM_THREADS) out[i] = -1;
    if (tid == 0 && n_sel) n_sel[row] = (int32_t)n;
}

int launch_glm_select(const float *scores, int batch, int64_t n_comp, int64_t npos, int kpool, int64_t topk,
                      int strict, int32_t *sel, int64_t max_sel, int32_t *n_sel, hipStream_t s) {
    CWICK_REQUIRE(scores && sel, "glm_select: null pointer");
    CWICK_REQUIRE(batch >= 1 && batch <= 65535 && n_comp >= 1 && n_comp <= ((int64_t)1 << 24),
                  "glm_select: batch %d, %lld pools", batch, (long long)n_comp);
    CWICK_REQUIRE(kpool >= 1 && kpool <= 8, "glm_select: kpool %d (1..8, src/attention.c:492)", kpool);
    CWICK_REQUIRE(topk >= 1 && topk <= 65536, "glm_select: topk %lld", (long long)topk);
    CWICK_REQUIRE(npos >= n_comp * kpool && npos < (n_comp + 1) * kpool,
                  "glm_select: %lld positions do not close exactly %lld pools of %d", (long long)npos,
                  (long long)n_comp, kpool);
    const int64_t want = (topk + kpool - 1) / kpool;
    CWICK_REQUIRE(max_sel >= (want + 1) * kpool && max_sel <= ((int64_t)1 << 24),
                  "glm_select: max_sel %lld (at least (ceil(topk / kpool) + 1) * kpool = %lld)", (long long)max_sel,
                  (long long)((want + 1) * kpool));
    if (n_comp <= want) {
        glm_expand_kernel<<<dim3(batch), GLM_THREADS, 0, s>>>(scores, nullptr, want, n_comp, npos, kpool, strict, 1, sel,
                                                            max_sel, n_sel);
        CWICK_HIP_CALL(hipGetLastError());
        return 1;
    }
    int32_t *pools = (int32_t *)workspace(s, (size_t)batch * want * sizeof(int32_t));
    if (!pools) return 0;                   // workspace() has recorded why
    if (!launch_topk(scores, batch, n_comp, want, pools, s)) return 0;
    glm_expand_kernel<<<dim3(batch), GLM_THREADS, 0, s>>>(scores, pools, want, n_comp, npos, kpool, strict, 0, sel,
                                                        max_sel, n_sel);
    CWICK_HIP_CALL(hipGetLastError());
    return 1;
}

int launch_candidate_apply(float *scores, const uint8_t *cand, int batch, int64_t n, hipStream_t s) {
    CWICK_REQUIRE(scores && cand && batch >= 1 && n >= 1, "candidate_apply: bad argument");
    const int64_t total = (int64_t)batch * n;
    int64_t blocks = (total + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    cand_apply_kernel<<<dim3((unsigned)blocks), 256, 0, s>>>(scores, cand, total);
    CWICK_HIP_CALL(hipGetLastError());
    return 1;
}

int launch_dequant_latent(const uint8_t *rows, const float *scales, int64_t n, float *out, hipStream_t s) {
    CWICK_REQUIRE(rows && scales && out && n > 0, "dequant_latent: bad argument");
    int64_t blocks = (n * CWICK_HIP_LATENT_KDIM + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    dequant_rows_kernel<CWICK_HIP_LATENT_KDIM, CWICK_HIP_LATENT_BLOCK><<<dim3((unsigned)blocks), 256, 0, s>>>(rows, scales, n, out);
    CWICK_HIP_CALL(hipGetLastError());
    return 1;
}

int launch_dequant_ikeys(const uint8_t *rows, const float *scales, int64_t n, float *out, hipStream_t s) {
    CWICK_REQUIRE(rows && scales && out && n > 0, "dequant_ikeys: bad argument");
    int64_t blocks = (n * CWICK_HIP_INDEX_DIM + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    dequant_rows_kernel<CWICK_HIP_INDEX_DIM, CWICK_HIP_INDEX_DIM><<<dim3((unsigned)blocks), 256, 0, s>>>(rows, scales, n, out);
    CWICK_HIP_CALL(hipGetLastError());
    return 1;
}

}  // namespace cwick
