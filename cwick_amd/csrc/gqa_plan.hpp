// gqa_plan.hpp -- how a chunk of the GQA prefill (gqa_prefill.hip) is dealt to workgroups.  Plain C++: the plan
// is made anew for every call, in front of kernels that may take 10 us, so it may not take long.
#pragma once
#include <stdint.h>

#include <initializer_list>

namespace cwick {

constexpr int PF_TK = 32;                   // keys of a tile
constexpr int PF_MAX_BLOCKS = 512;
// The position blocks of a chunk and the slices that their keys are cut into, a workgroup each (and one of each
// for every kv head).  Rank 0 is the last block; block rank r has slices first[r] .. first[r + 1], of `per`
// tiles each, the last one with the rest of the block.  per = 0: whole blocks.
struct PfPlan {
    int per;
    uint16_t first[PF_MAX_BLOCKS + 1];
};

// keys a block of `positions` positions attends to: 0 .. its last position (clipped to the chunk)
__host__ __device__ inline int64_t pf_keys(int64_t pos0, int64_t n, int positions, int64_t pblk) {
    const int64_t last = (pblk + 1) * positions;
    return pos0 + (last < n ? last : n);
}
// Slices of a block of `tiles` tiles whose first `plain` need no mask: as many as `per` fit, every
// slice beginning below the diagonal (the first tile of a slice must give every row its reference).
__host__ __device__ inline int pf_slices(int tiles, int plain, int per) {
    const int by_tiles = (int)((uint32_t)(tiles + per - 1) / (uint32_t)per), by_plain = 1 + (int)((uint32_t)plain / (uint32_t)per);
    return by_tiles < by_plain ? by_tiles : by_plain;
}

// What a kernel's workgroups take, in microseconds: the launch, a workgroup besides its tiles, a step of
// `waves` tiles (with two-term weights; what it takes longer when every compute unit is at work all the time),
// and, where there are slices, the second launch, more for each slice of a block, and each slice's partials
// (written and read).  Fitted to 150 times of 21 shapes for the first and 170 of 52 for the second (16 to 8192
// positions behind 0 to 16000, between none and sixty slices); the times of list scheduling with these
// figures are 3.4 and 5.5 % off them (rms).
struct PfCost {
    int waves, least;                       // tiles of a step; the fewest tiles of a slice
    float launch, item, step, step2, crowd, merge, merge_slice, merge_part;
};
constexpr PfCost PF_COST_WIDE = {1, 4, 7.0f, 5.0f, 1.19f, 2.19f, 0.45f, 3.7f, 0.05f, 0.085f};       // 256 rows
constexpr PfCost PF_COST_TEAM = {4, 4, 2.3f, 7.1f, 1.64f, 2.3f, 0.46f, 2.2f, 0.065f, 0.023f};       // 64 rows

struct PfBlocks {
    int count, n_kv_heads, n_prec, cus;     // the first n_prec blocks take two-term weights
    int tiles[PF_MAX_BLOCKS], plain[PF_MAX_BLOCKS];     // by rank
};

// The time of a plan, or anything from `limit` on where it takes at least that, and its slices of blocks that are
// cut.  The kernels hand their workgroups out in the order of the ranks, each to the compute unit that is
// free first.
inline float pf_time(const PfBlocks &b, const PfCost &c, int per, float limit, int &parts) {
    int items = 0, most = 1;
    parts = 0;
    uint16_t cut[PF_MAX_BLOCKS];            // slices of each block
    for (int r = 0; r < b.count; r++) {
        const int k = per && b.tiles[r] > per ? pf_slices(b.tiles[r], b.plain[r], per) : 1;
        cut[r] = (uint16_t)k;
        items += k;
        if (k > 1) parts += k;
        if (k > most) most = k;
    }
    const int n = items * b.n_kv_heads;
    const float end = parts ? c.merge + c.merge_slice * (float)most + c.merge_part * (float)(parts * b.n_kv_heads) : 0.0f;
    auto steps = [&](int tiles) { return (float)(c.waves == 1 ? tiles : (tiles + 3) / 4); };
    auto step = [&](int r) { return b.count - 1 - r < b.n_prec ? c.step2 : c.step; };
    float sum = 0.0f, sum_steps = 0.0f, longest = 0.0f, longest_steps = 0.0f;
    auto add = [&](int r, int tiles, int times) {
        const float x = steps(tiles), t = c.item + step(r) * x;
        sum += t * (float)times;
        sum_steps += x * (float)times;
        if (t > longest) longest = t, longest_steps = x;
    };
    for (int r = 0; r < b.count; r++) {
        const int k = cut[r];
        add(r, b.tiles[r] - (k - 1) * per, 1);
        if (k > 1) add(r, per, k - 1);
    }
    const float share = (float)b.n_kv_heads / (float)b.cus;
    const float crowd = c.crowd * (sum * share < longest ? sum * share / longest : 1.0f);
    const float even = (sum + crowd * sum_steps) * share, alone = longest + crowd * longest_steps;
    const float least = even > alone ? even : alone;
    auto cost = [&](int r, int tiles) { return c.item + (step(r) + crowd) * steps(tiles); };
    if (n <= b.cus || c.launch + least + end >= limit) return c.launch + least + end;
    // list scheduling, the kv heads of a slice as one where they go into the compute units evenly
    const bool joint = b.cus % b.n_kv_heads == 0;
    const int machines = joint ? b.cus / b.n_kv_heads : b.cus, copies = joint ? 1 : b.n_kv_heads;
    float heap[1024];                       // when each is free, the first to be at the top
    if (machines > 1024) return c.launch + least + end;
    int used = 0;
    float last = 0.0f;
    auto deal = [&](float t) {
        if (used < machines) {              // one that has had nothing yet (the heap is made when there is none left)
            heap[used++] = t;
            last = t > last ? t : last;
            if (used < machines) return;
            for (int i = machines / 2 - 1; i >= 0; i--) {
                const float v = heap[i];
                int j = i;
                for (int ch; (ch = 2 * j + 1) < machines; j = ch) {
                    if (ch + 1 < machines && heap[ch + 1] < heap[ch]) ch++;
                    if (heap[ch] >= v) break;
                    heap[j] = heap[ch];
                }
                heap[j] = v;
            }
            return;
        }
        const float v = heap[0] + t;
        last = v > last ? v : last;
        int j = 0;
        for (int ch; (ch = 2 * j + 1) < machines; j = ch) {
            if (ch + 1 < machines && heap[ch + 1] < heap[ch]) ch++;
            if (heap[ch] >= v) break;
            heap[j] = heap[ch];
        }
        heap[j] = v;
    };
    for (int r = 0; r < b.count && c.launch + last + end < limit; r++) {
        const int k = cut[r];
        const float rest = cost(r, b.tiles[r] - (k - 1) * per), full = k > 1 ? cost(r, per) : rest;
        for (int i = 0; i < k; i++)
            for (int x = 0; x < copies; x++) deal(i + 1 < k ? full : rest);
    }
    return c.launch + last + end;
}

// The best plan of one kernel for a chunk whose blocks have `positions` positions each (at most PF_MAX_BLOCKS of
// them, n_prec with two-term weights), if it takes less than `limit`: its time, else `limit`.
// Tried are whole blocks; the shortest slices that every compute unit gets at most one of, and slices longer
// by a quarter to three times (fewer partials); where they are long, those for two and three rounds (for blocks
// of about the same length, also behind the rounds that whole blocks take); and, where there is half a round of whole blocks to one and a
// half, slices that cut only the last blocks in two.
inline float pf_plan(int64_t pos0, int64_t n, int positions, int n_kv_heads, int64_t n_prec, int cus, const PfCost &c,
                     float limit, PfPlan &best) {
    PfBlocks b;
    b.count = (int)((n + positions - 1) / positions);
    // (the even share of all tiles with one-term weights: nothing takes less)
    const float keys = (float)b.count * (float)pos0 + 0.5f * (float)n * (float)b.count;
    if (c.launch + ((float)b.count * c.item + keys / (float)(PF_TK * c.waves) * c.step) * (float)n_kv_heads / (float)cus >= limit) return limit;
    b.n_kv_heads = n_kv_heads;
    b.n_prec = (int)n_prec;
    b.cus = cus;
    int64_t total = 0;
    for (int r = 0; r < b.count; r++) {
        const int64_t pb = b.count - 1 - r;
        b.tiles[r] = (int)((uint32_t)(pf_keys(pos0, n, positions, pb) + PF_TK - 1) / PF_TK);      // (at most 2^30 keys)
        b.plain[r] = (int)((uint32_t)(pos0 + pb * positions + 1) / PF_TK);
        total += b.tiles[r];
    }
    const int most = b.tiles[0];
    float best_t = limit;
    int best_per = -1;
    int best_parts = 0;
    // (Of two plans within 2 % the one with fewer slices: 700 positions behind 12000 take 157 us in 220 slices and
    // 159 to 171, for the same by these figures, in 244.)
    auto look = [&](int per) {
        if (per && (per < c.least || per >= most)) return;
        int parts;
        const float t = pf_time(b, c, per, 1.02f * best_t, parts);
        if (t < limit && (best_per < 0 ? t < best_t : parts < best_parts ? t < 1.02f * best_t : t < 0.98f * best_t))
            best_t = t, best_per = per, best_parts = parts;
    };
    look(0);
    const int room = cus / n_kv_heads;      // slices for one round
    // (A prompt of one round of whole blocks, at the beginning of a cache, stays whole and takes no memory for partials:
    // 4096 positions of 16 / 4 heads 176 us, cut 164; 8192 of 8 / 8 330 and 275.  Behind earlier keys it is a chunk
    // like its neighbours, whole and cut: 4096 of 16 / 4 behind 500 keys 207 and 195, 2048 295 and 274, 4096 402 and
    // 370, 8192 615 and 595; of 16 / 2 behind 2048 292 and 260; 8192 of 8 / 8 behind 2048 510 and 377.)
    const bool whole = pos0 == 0 && b.count == room;
    if (!whole && (b.count < room || (room > 0 && 2 * b.tiles[b.count - 1] > most))) {
        auto round_up = [&](int64_t per) { return (int)(c.waves == 1 ? per : (per + 3) / 4 * 4); };
        const int first = b.count / room + 1;
        for (int rounds = first; rounds < first + 3; rounds++) {
            int fit = round_up((total + rounds * room - 1) / (rounds * room));
            if (rounds > 1 && fit <= 12 * c.waves) break;       // (a round more costs as much as six steps)
            fit = fit < c.least ? c.least : fit;
            auto fits = [&](int per) {
                int items = 0;
                for (int r = 0; r < b.count; r++) items += b.tiles[r] > per ? pf_slices(b.tiles[r], b.plain[r], per) : 1;
                return items <= rounds * room;
            };
            while (!fits(fit)) fit = round_up(fit + 1 + fit / 16);
            for (int back = fit / 16; back > 0 && fit - c.waves >= c.least && fits(fit - c.waves); back -= c.waves) fit -= c.waves;
            look(fit);
            const int cuts = pf_slices(most, b.plain[0], fit);      // one slice fewer for the longest block, if that is even
            if (cuts > 1 && cuts < 12) look(round_up((most + cuts - 2) / (cuts - 1)));
            if (rounds == 1)
                for (int quarters : {5, 6, 8, 12}) look(round_up((int64_t)fit * quarters / 4));
        }
    }
    if (!whole && 2 * b.count >= room && 2 * b.count <= 3 * room)
        for (int eighths : {7, 6, 5, 4}) look((most * eighths + 7) / 8);
    if (best_per < 0) return limit;
    best.per = best_per;
    best.first[0] = 0;
    for (int r = 0; r < b.count; r++)
        best.first[r + 1] = (uint16_t)(best.first[r] + (best_per ? pf_slices(b.tiles[r], b.plain[r], best_per) : 1));
    if (best.first[1] == 1) best.per = 0;   // (slices longer than any block)
    return best_t;
}

}  // namespace cwick
