// mla_plan.hpp -- how a chunk of the latent prefill (mla_prefill64.hip) and a latent decode (mla_roles.hip) are dealt
// to workgroups.  Plain C++: a plan is made anew for every call, in front of kernels that may take 10 us, so it may
// not take long.
#pragma once
#include <stdint.h>

namespace cwick {

// Row blocks (sixteen heads of a query) come in groups of four, two or one, a workgroup each.  The last
// `whole` groups, which have the most keys, take all of theirs; the keys of the others are cut into
// `slices` slices, a workgroup each.
// One workgroup runs per compute unit, so whole groups beyond the last full round leave units idle; cut,
// they fill it.  In steps of one key tile (1.45 us) a workgroup costs its tiles and five more (Q, the
// first tiles' way into LDS, the output; three and two for smaller groups); the merge costs three and a
// hundredth per slice, the partials one for every 256 row blocks (32 KB each, written and read); and when
// every compute unit is busy the clock drops by a sixth, so a round that is not full is cheaper than its
// share.  Fitted to a sweep of group sizes and slice counts over 25 shapes (1 to 512 queries of 16 to 128
// heads behind 200 to 28000 rows): what it picks is 0.7 % slower than the best of the sweep on the mean,
// 7 % at the worst.  333 queries of 64 heads over 1624 rows 86 us whole, 80 with the last 77 groups in
// three slices; 180 groups of 2090 rows 58 us whole, 81 in two slices; 20 queries of 64 heads over 320
// rows 13.8 us in groups of one row block, 21 in five slices of groups of two.
struct WidePlan {
    uint32_t gsz, groups, whole, slices;
    float time;
};

// the time of `wgs` workgroups of `tiles` tiles (up to four rounds of them)
inline float plan_rounds(int wgs, int tiles, float over, int cus, float cu) {      // cu: 1 / cus
    const int full = (wgs >= cus) + (wgs >= 2 * cus) + (wgs >= 3 * cus) + (wgs >= 4 * cus), left = wgs - full * cus;
    const float last = 1.2f * (float)left * cu;
    return ((float)full * 1.2f + (left == 0 ? 0.0f : last < 1.0f ? 1.0f : last)) * ((float)tiles + over);
}
inline float plan_over(int gsz) { return gsz == 4 ? 5.0f : gsz == 2 ? 3.0f : 2.0f; }
// the time of `rest` groups in s slices of up to `per` tiles each
inline float plan_sliced(int gsz, int rest, int per, int s, int cus, float cu) {
    return 3.0f + 0.01f * (float)s + (float)(gsz * rest * s) * cu + plan_rounds(rest * s, per, plan_over(gsz), cus, cu);
}

// The best plan for groups of one size.  tiles_first and tiles_last: key tiles of the chunk's first and last query.
inline WidePlan plan_slices(int64_t n_rb, int gsz, int64_t tiles_first, int64_t tiles_last, int cus) {
    const int64_t groups = (n_rb + gsz - 1) / gsz;
    const float over = plan_over(gsz), cu = 1.0f / (float)cus;
    WidePlan best{(uint32_t)gsz, (uint32_t)groups, (uint32_t)groups, 1, 0.0f};
    if (groups > 16 * (int64_t)cus) return best;     // many rounds: what the last one leaves idle is nothing
    auto tiles_at = [&](int64_t i) { return (int)(tiles_first + (tiles_last - tiles_first) * i / (groups > 1 ? groups - 1 : 1)); };
    auto whole_time = [&](int whole) {               // whole groups from the last one down
        float t = 0.0f;
        for (int done = 0; done < whole; done += cus)
            t += plan_rounds(whole - done < cus ? whole - done : cus, tiles_at(groups - 1 - done), over, cus, cu);
        return t;
    };
    best.time = whole_time((int)groups);
    const int full = (int)groups / cus * cus;
    for (int whole = full; whole >= 0 && whole >= full - cus; whole -= cus) {
        const int rest = (int)groups - whole, tiles = rest ? tiles_at(rest - 1) : 0;
        if (!rest) continue;
        const float base = whole_time(whole);
        const int most = tiles < 4 * cus / rest ? tiles : 4 * cus / rest;
        // Slices of as many tiles each: the fewest of them are the best.  So a slice count stands for its tiles
        // per slice; counts go up in steps of a quarter, and then the tiles per slice around the best are
        // tried one by one.  No count is better once the partials and the least a round costs are too much.
        float best_t = 1e30f;
        int best_per = 0;
        auto look = [&](int per) {
            const int s = (tiles + per - 1) / per;
            if (s < 2 || s > most) return;
            const float t = base + plan_sliced(gsz, rest, per, s, cus, cu);
            if (t < best_t) best_t = t, best_per = per;
        };
        for (int s = 2, last_per = 0; s <= most; s = s < 8 ? s + 1 : s + s / 4) {
            if (base + 3.0f + (float)(gsz * rest * s) * cu + over >= (best_t < best.time ? best_t : best.time)) break;
            const int per = (tiles + s - 1) / s;
            if (per != last_per) look(per);
            last_per = per;
        }
        if (!best_per) continue;
        const int mid = best_per, around = mid / 5 < 6 ? mid / 5 + 1 : 6;
        for (int d = 1; d <= around; d++) {
            if (mid > d) look(mid - d);
            look(mid + d);
        }
        // the count that fills the round
        const int fill = cus / rest;
        if (fill >= 2 && fill <= most) look((tiles + fill - 1) / fill);
        if (best_t < best.time) best.whole = (uint32_t)whole, best.slices = (uint32_t)((tiles + best_per - 1) / best_per), best.time = best_t;
    }
    return best;
}

inline WidePlan plan_wide(int64_t n_rb, int64_t tiles_first, int64_t tiles_last, int cus) {
    WidePlan best = plan_slices(n_rb, 4, tiles_first, tiles_last, cus);
    for (int gsz = 2; gsz >= 1 && (n_rb + gsz - 1) / gsz <= cus; gsz /= 2) {
        const WidePlan x = plan_slices(n_rb, gsz, tiles_first, tiles_last, cus);
        if (x.time < best.time) best = x;
    }
    return best;
}

// The decode: how many slices the keys of one query can be cut into.  `blocks` are its blocks of 32 heads, of all
// queries; one workgroup is resident per compute unit (per_cu: more are asked for), so one round of them at most.
constexpr int MLA_MAX_SPLITS = 1024;
inline int64_t mla_decode_most_splits(int64_t blocks, int per_cu, int cus) {
    const int64_t want = (int64_t)per_cu * cus / blocks;
    return want < 1 ? 1 : want > MLA_MAX_SPLITS ? MLA_MAX_SPLITS : want;
}
// The tiles of 64 keys of a workgroup.  With up to three of them each, fewer workgroups of a tile or more in addition
// are often the shorter ones: a further tile takes 1.1 us (out of a list 1.5), while all workgroups start, write their
// partials and have them merged at the same time, 2.5 us for 128 of them and 6.2 for 256 (fitted to 150 times when a step took
// 2 800 cycles, now 2 200; left alone from four tiles on, where the end of the workgroups spreads).  Of the kernels as they are, 250
// shapes: 0.7 % behind the fastest number of tiles on the mean, 11 % at the worst (8 lists of 1280 rows for 48 heads); a full
// round 1.9 % and 17.  us, replayed from a graph, with the workgroups of a full round and as chosen here: 64 heads, 8192 keys
// 15.1 and 12.1, 16384 16.2 and 14.0; 128 heads, 4096 14.3 and 11.9, 12288 16.1 and 15.4; 16 heads, 32768 16.1 and 14.4; 8 x 600
// keys of 64 heads 12.6 and 11.1; 4 x 2048 out of lists of 64 heads 14.7 and 12.5; equal where it is closest, 2 x 12000 of 64.
// Two tiles in one workgroup take less than the merge (100 keys of 16 heads: 8.3 and 7.4).
inline int64_t mla_decode_tiles(int64_t tiles, int64_t blocks, bool list, int per_cu, int cus) {
    const int64_t want = mla_decode_most_splits(blocks, per_cu, cus);
    int64_t per = (tiles + want - 1) / want;
    if (per_cu != 1) return per;                            // (as many as that makes)
    if (tiles <= 2) return tiles;
    if (per > 3) return per;
    const float step = list ? 1.5f : 1.1f;
    float best = 1e30f;
    for (int64_t t = per, end = per + 3; t <= end; t++) {
        const float wgs = (float)((tiles + t - 1) / t * blocks), cost = step * (float)t + (0.014f + 4e-5f * wgs) * wgs;
        if (cost < best) best = cost, per = t;
    }
    return per;
}

}  // namespace cwick
