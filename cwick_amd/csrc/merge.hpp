// merge.hpp -- second pass of split-K flash-decoding: combine the per-slice
// partials (m_s, l_s, acc_s) of one query row into the normalised output
//
//     out[d] = sum_s acc_s[d] 2^{m_s - M} / sum_s l_s 2^{m_s - M},  M = max_s m_s.
//
// One workgroup per (head, query).
#pragma once
#include "common.hpp"

#include <type_traits>

namespace cwick {

// One workgroup per (head, query), a wave per slice up to sixteen; wave w takes slices w, w + n_waves, ... (up to eight
// at a time), lane = one float4 of the row; the waves meet in LDS.
// The chain is one trip to memory and the meeting, so every load goes out before anything is waited for: as many as
// the slices need, past the last one that one again, without a branch between them.  The maximum and the sum of
// slice j of the eight come to lanes with lane % 8 = j in one load (a load of one address for all lanes takes the memory
// pipeline as long as a row does) and go to the others through scalar registers.  (Under a branch each, with scalar
// loads in them, the loads waited for one another.  64 slices of 16 heads x 256: 3.8 us, now 3.4; 4096 keys 10.1, 9.75;
// 12000 of 64 heads x 128 on 4 11.6, 10.9.)
template <int DIM>
__global__ void __launch_bounds__(1024)
splitk_merge_wide_kernel(const float *__restrict__ part_acc,   // [y][split][head][DIM]
                         const float *__restrict__ part_ml,    // [y][split][head][2]
                         int n_splits, int n_heads, float *__restrict__ out /* [y][head][DIM] */,
                         uint32_t *flags, uint32_t epoch) {               // one flag per head, or null
    static_assert(DIM % 4 == 0 && DIM <= 256, "one float4 per lane");
    __shared__ float red_m[16];
    __shared__ float red_l[16];
    __shared__ f32x4 red_a[16][64];
    const int h = blockIdx.x, y = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), mw = n_splits < 16 ? n_splits : 16;     // the launch's waves
    const bool live = lane < DIM / 4;
    const size_t base = (size_t)y * n_splits;
    const float *ml = part_ml + (base * n_heads + h) * 2;
    const uint32_t ml_stride = (uint32_t)n_heads * 2;
    const float *pa = part_acc + (base * n_heads + h) * DIM + (live ? lane : 0) * 4;
    const uint32_t pa_stride = (uint32_t)n_heads * DIM;

    f32x4 a[8];
    f32x2 v;                                            // of slice s0 + mw (lane % 8); none: -inf, 0
    auto fetch = [&](int s0, auto count) {
        const int sl = s0 + mw * (lane & 7);
        v = *(const f32x2 *)(ml + (size_t)(sl < n_splits ? sl : n_splits - 1) * ml_stride);
#pragma unroll
        for (int j = 0; j < decltype(count)::value; j++) {
            const int s = s0 + mw * j;
            a[j] = *(const f32x4 *)(pa + (size_t)(s < n_splits ? s : n_splits - 1) * pa_stride);
        }
        if (sl >= n_splits) v = (f32x2){-INFINITY, 0.0f};
    };
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    float ls = 0.f, mx = -INFINITY;                     // ls: over this lane's slices
    auto add = [&](auto count) {
        const float c = v[0] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(v[0] - mx);
        ls = __builtin_fmaf(v[1], c, ls);
#pragma unroll
        for (int j = 0; j < decltype(count)::value; j++) {
            const float cj = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, c), j));
#pragma unroll
            for (int r = 0; r < 4; r++) acc[r] = __builtin_fmaf(a[j][r], cj, acc[r]);
        }
    };
    // the largest maximum of all waves
    auto meet = [&] {
        mx = row_max(mx);
        if (lane == 0) red_m[wv] = mx;
        __syncthreads();
        mx = row_max((lane & 15) < mw ? red_m[lane & 15] : -INFINITY);
    };
    auto few = [&](auto count) {
        fetch(wv, count);
        mx = v[0];
        meet();
        add(count);
    };
    if (n_splits <= 16) few(std::integral_constant<int, 1>{});
    else if (n_splits <= 64) few(std::integral_constant<int, 4>{});
    else if (n_splits <= 128) few(std::integral_constant<int, 8>{});
    else {
        const std::integral_constant<int, 8> eight;
        fetch(wv, eight);
        mx = v[0];
        for (int s = wv + mw * (8 + (lane & 7)); s < n_splits; s += 8 * mw) mx = fmaxf(mx, ml[(size_t)s * ml_stride]);
        meet();
        add(eight);
        for (int s0 = wv + 8 * mw; s0 < n_splits; s0 += 8 * mw) {
            fetch(s0, eight);
            add(eight);
        }
    }
    ls = group_step_sum<8>(group_step_sum<4>(group_step_sum<2>(ls)));
    if (lane == 0) red_l[wv] = ls;
    red_a[wv][lane] = acc;
    __syncthreads();
    if (wv != 0 || !live) return;
    float l = 0.f;
    f32x4 r4 = {0.f, 0.f, 0.f, 0.f};
    if (mw == 16) {
        f32x4 t[16];
#pragma unroll
        for (int w = 0; w < 16; w++) t[w] = red_a[w][lane];
#pragma unroll
        for (int w = 0; w < 16; w++) {
            l += red_l[w];
#pragma unroll
            for (int r = 0; r < 4; r++) r4[r] += t[w][r];
        }
    } else {
        for (int w = 0; w < mw; w++) {
            l += red_l[w];
            const f32x4 t = red_a[w][lane];
#pragma unroll
            for (int r = 0; r < 4; r++) r4[r] += t[r];
        }
    }
    const float inv = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
    for (int r = 0; r < 4; r++) r4[r] *= inv;
    float *dst = out + ((size_t)y * n_heads + h) * DIM + lane * 4;
    if (!flags) {
        *(f32x4 *)dst = r4;
    } else {                                            // (one wave writes the head)
        store_through16(dst, __builtin_bit_cast(u32x4, r4));
        stores_done();
        if (lane == 0) host_flag(flags, h, epoch);
    }
}

}  // namespace cwick
