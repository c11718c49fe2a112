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
// `waves` tiles (with two-term weights; what it takes longer where every compute unit of its XCD is at work all the
// time, and from which share of them on it takes longer at all), and, where there are slices, the second launch, more
// for each slice of a block, and each slice's partials (written and read).
// Fitted to 20500 times of 1049 shapes (1 to 8192 positions behind 0 to 16000 of one to eight heads on one to
// eight kv heads, whole and in slices) when workgroups of few steps had no body of their own; its prices (few_*) came with it, the
// others stayed.  12791 times of 984 such shapes, of the kernels as they are: of the plans of a shape the one with the least price
// is 0.5 % behind the fastest on the mean, 15 % at the worst (129 positions at the beginning of 16 / 4 heads, cut in two and
// whole: 13.1 and 11.4 us) but for six kv heads (84 behind 13135 of 12 / 6: 47.8, in slices an eighth longer 34.4).  The prices of
// plans near the fastest are 4.0 % off (rms) with 256 rows, with 64 rows 3.2 in slices of more steps, 8.4 of few, and 25 for
// whole blocks, whose calls of 8 to 15 us they have 14 % too long on the mean.
// What counts is the share of an XCD's own units that are at work, and up to a third or a half of them it adds nothing:
// 1.21 us a tile with up to half of them, 1.33 with 64 %, 1.55 with 90.  With the mean of the chip, and in
// proportion from the first unit on, two slices a block (the long ones of which lie on half of the XCDs, where there
// are four kv heads) looked shorter than four, and whole blocks of 64 rows shorter than slices: 2500 positions
// behind 4000 of 16 / 4 heads 287 us, now 252; 2800 298, 271; 4000 of 8 / 8 240, 211.
struct PfCost {
    int waves, least;                       // tiles of a step; the fewest tiles of a slice
    float launch, item, step, step2, crowd, alone, merge, merge_slice, merge_part;
    // workgroups of up to `few` steps (`few2` with two-term weights), where another body is the shorter one
    int few, few2;
    float few_item, few_step, few_step2;
};
// Steps of a workgroup up to which that is so: where the prices below cross.  (Four and five steps with two-term weights, in
// that body and the other: 500 positions of 32 / 4 heads 20.7 and 19.8 us, 560 24.1 and 23.1, 411 behind 210 23.4 and 22.0,
// 236 of 64 / 8 behind 334 23.4 and 22.2; seven with one-term weights the same to 0.5 %: 100 behind 7000 27.4 and 27.5.)
constexpr int PF_ROUNDS = 6, PF_ROUNDS2 = 3;
constexpr PfCost PF_COST_WIDE = {1, 4, 0.8f, 9.6f, 1.22f, 2.135f, 0.411f, 0.36f, 4.8f, 0.021f, 0.063f, 0, 0, 0.0f, 0.0f, 0.0f};      // 256 rows
constexpr PfCost PF_COST_TEAM = {4, 4, 2.5f, 7.25f, 1.815f, 2.46f, 0.362f, 0.44f, 2.5f, 0.072f, 0.016f, PF_ROUNDS, PF_ROUNDS2, 3.9f, 2.3f, 3.3f};      // 64 rows
constexpr bool pf_crosses(int steps, float few_step, float step) {
    const PfCost &c = PF_COST_TEAM;
    return c.few_item + few_step * (float)steps <= c.item + step * (float)steps && c.few_item + few_step * (float)(steps + 1) > c.item + step * (float)(steps + 1);
}
static_assert(pf_crosses(PF_ROUNDS, PF_COST_TEAM.few_step, PF_COST_TEAM.step) && pf_crosses(PF_ROUNDS2, PF_COST_TEAM.few_step2, PF_COST_TEAM.step2),
              "the limits of the other body are not where its prices end to be the lesser ones");

struct PfBlocks {
    int count, n_kv_heads, n_prec, cus;     // the first n_prec blocks take two-term weights
    int tiles[PF_MAX_BLOCKS], plain[PF_MAX_BLOCKS];     // by rank
};

// What a plan comes to: its slices of each block, how many of them belong to blocks that are cut, the time of their
// merge, and with their sums the least time: the even share or the longest, with the units of all XCDs at
// work alike (seldom more than it is).
struct PfSums {
    int items, parts;
    float end, sum, sum_steps, least;
    uint16_t cut[PF_MAX_BLOCKS];
};
inline float pf_steps(const PfCost &c, int tiles) { return (float)(c.waves == 1 ? tiles : (tiles + 3) / 4); }
inline float pf_slice_time(const PfBlocks &b, const PfCost &c, int r, int tiles) {
    const bool two = b.count - 1 - r < b.n_prec;
    const float steps = pf_steps(c, tiles);
    return steps <= (float)(two ? c.few2 : c.few) ? c.few_item + (two ? c.few_step2 : c.few_step) * steps : c.item + (two ? c.step2 : c.step) * steps;
}
// what a step takes longer, from the share of the units at work when they start and the mean of it: it falls evenly
inline float pf_slower(const PfCost &c, float at_first, float mean) {
    const float at_last = 2.0f * mean - at_first, room = 1.0f - c.alone;
    if (at_last >= c.alone || at_first <= at_last) return mean > c.alone ? c.crowd * (mean < 1.0f ? mean - c.alone : room) / room : 0.0f;
    if (at_first <= c.alone) return 0.0f;
    const float over = at_first - c.alone;
    return c.crowd * over * over / (2.0f * (at_first - at_last) * room);
}
inline void pf_sums(const PfBlocks &b, const PfCost &c, int per, PfSums &p) {
    int most = 1;
    float longest = 0.0f, longest_steps = 0.0f;
    const float full_steps = pf_steps(c, per);
    p.items = p.parts = 0;
    p.sum = p.sum_steps = 0.0f;
    for (int r = 0; r < b.count; r++) {
        const int k = per && b.tiles[r] > per ? pf_slices(b.tiles[r], b.plain[r], per) : 1, left = b.tiles[r] - (k - 1) * per;
        const float rest = pf_slice_time(b, c, r, left), rest_steps = pf_steps(c, left);
        p.cut[r] = (uint16_t)k;
        p.items += k;
        p.sum += rest;
        p.sum_steps += rest_steps;
        if (rest > longest) longest = rest, longest_steps = rest_steps;
        if (k == 1) continue;
        const float full = pf_slice_time(b, c, r, per);
        p.parts += k;
        p.sum += full * (float)(k - 1);
        p.sum_steps += full_steps * (float)(k - 1);
        if (k > most) most = k;
        if (full > longest) longest = full, longest_steps = full_steps;
    }
    p.end = p.parts ? c.merge + c.merge_slice * (float)most + c.merge_part * (float)(p.parts * b.n_kv_heads) : 0.0f;
    const float part_of = (float)b.n_kv_heads / (float)b.cus, even = p.sum * part_of;
    const float x = pf_slower(c, (float)p.items * part_of < 1.0f ? (float)p.items * part_of : 1.0f, even / longest);
    const float even_x = even + x * p.sum_steps * part_of, longest_x = longest + x * longest_steps;
    p.least = c.launch + (even_x > longest_x ? even_x : longest_x) + p.end;
}

// The time of a plan, or anything from `limit` on where it takes at least that.  The kernels hand their workgroups out
// in the order of the ranks, the first to the XCDs in turn and the others each to the compute unit that is free first.
inline float pf_time(const PfBlocks &b, const PfCost &c, int per, const PfSums &p, float limit) {
    const bool joint = b.cus % b.n_kv_heads == 0;       // the kv heads of a slice as one where they go into the units evenly
    const int machines = joint ? b.cus / b.n_kv_heads : b.cus, copies = joint ? 1 : b.n_kv_heads;
    const int kv = b.n_kv_heads, groups = !joint || kv % 8 == 0 ? 1 : kv % 4 == 0 ? 2 : kv % 2 == 0 ? 4 : 8;
    const bool at_once = p.items * copies <= machines;
    if (machines > 1024 || (at_once && groups == 1)) return p.least;
    // what the XCDs of each group (those of the slices with its remainder) do, and until when
    float busy[8] = {}, last[8] = {}, start[8] = {};
    if (at_once) {
        int i = 0;
        for (int g = 0; g < groups; g++) start[g] = (float)((p.items - g + groups - 1) / groups * groups) / (float)machines;
        for (int r = 0; r < b.count; r++) {
            const int k = p.cut[r];
            const float rest = pf_slice_time(b, c, r, b.tiles[r] - (k - 1) * per), full = k > 1 ? pf_slice_time(b, c, r, per) : 0.0f;
            for (int g = 0; g < groups && g < k - 1; g++) {
                const int to = (i + g) % groups;
                busy[to] += full * (float)((k - 2 - g) / groups + 1);
                last[to] = full > last[to] ? full : last[to];
            }
            i += k;
            const int to = (i - 1) % groups;
            busy[to] += rest;
            last[to] = rest > last[to] ? rest : last[to];
        }
    } else {
        // list scheduling
        for (int g = 0; g < groups; g++) start[g] = 1.0f;
        float free_at[1024], latest = 0.0f;             // the first to be free at the top, once each has had a slice
        uint8_t of[1024];
        int used = 0;
        auto sink = [&](int at) {
            const float v = free_at[at];
            const uint8_t g = of[at];
            int j = at;
            for (int ch; (ch = 2 * j + 1) < machines; j = ch) {
                if (ch + 1 < machines && free_at[ch + 1] < free_at[ch]) ch++;
                if (free_at[ch] >= v) break;
                free_at[j] = free_at[ch];
                of[j] = of[ch];
            }
            free_at[j] = v;
            of[j] = g;
        };
        auto deal = [&](float t) {
            const bool first = used < machines;
            const int at = first ? used : 0;
            if (first) free_at[at] = 0.0f, of[at] = (uint8_t)(used % groups);
            const float until = free_at[at] + t;
            const int g = of[at];
            free_at[at] = until;
            busy[g] += t;
            last[g] = until > last[g] ? until : last[g];
            latest = until > latest ? until : latest;
            if (!first) sink(0);
            else if (++used == machines)
                for (int i = machines / 2 - 1; i >= 0; i--) sink(i);
        };
        for (int r = 0; r < b.count && c.launch + latest + p.end < limit; r++) {
            const int k = p.cut[r];
            const float rest = pf_slice_time(b, c, r, b.tiles[r] - (k - 1) * per), full = k > 1 ? pf_slice_time(b, c, r, per) : 0.0f;
            for (int i = 0; i < k; i++)
                for (int n = 0; n < copies; n++) deal(i + 1 < k ? full : rest);
        }
    }
    float t = 0.0f;
    for (int g = 0; g < groups; g++) {
        if (last[g] == 0.0f) continue;
        const float until = last[g] * (1.0f + pf_slower(c, start[g], busy[g] * (float)groups / ((float)machines * last[g])) * p.sum_steps / p.sum);
        t = until > t ? until : t;
    }
    return c.launch + t + p.end;
}

// the same with the sums of the plan, and its slices of blocks that are cut
inline float pf_time(const PfBlocks &b, const PfCost &c, int per, float limit, int &parts) {
    PfSums p;
    pf_sums(b, c, per, p);
    parts = p.parts;
    return p.least >= limit ? p.least : pf_time(b, c, per, p, limit);
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
    if (c.launch + ((float)b.count * (c.few ? c.few_item : c.item) + keys / (float)(PF_TK * c.waves) * c.step) * (float)n_kv_heads / (float)cus >= limit) return limit;
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
    // the plans to try: their slice lengths, and what each takes at least
    int tries = 0, pers[24];
    float least[24];
    PfSums sums;
    auto look = [&](int per) {
        if ((per && (per < c.least || per >= most)) || tries == 24) return;
        for (int i = 0; i < tries; i++)
            if (pers[i] == per) return;
        pf_sums(b, c, per, sums);
        if (per && sums.items * n_kv_heads > 4 * cus) return;   // (memory for the partials: 258 MiB for 1024 slices of 256 rows)
        pers[tries] = per;
        least[tries++] = sums.least;
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
                for (int r = 0; r < b.count && items <= rounds * room; r++) items += b.tiles[r] > per ? pf_slices(b.tiles[r], b.plain[r], per) : 1;
                return items <= rounds * room;
            };
            while (!fits(fit)) fit = round_up(fit + 1 + fit / 16);
            for (int back = fit / 16; back > 0 && fit - c.waves >= c.least && fits(fit - c.waves); back -= c.waves) fit -= c.waves;
            look(fit);
            const int cuts = pf_slices(most, b.plain[0], fit);      // as many even slices for the longest block, and one fewer
            if (cuts > 1 && cuts < 12) look(round_up((most + cuts - 1) / cuts)), look(round_up((most + cuts - 2) / (cuts - 1)));
            if (rounds == 1)
                for (int quarters : {5, 6, 8, 12}) look(round_up((int64_t)fit * quarters / 4));
        }
    }
    if (!whole && 2 * b.count >= room && 2 * b.count <= 3 * room)
        for (int eighths : {7, 6, 5, 4}) look((most * eighths + 7) / 8);
    // The ones that may be the shortest first.  (Of the plans within 2 % of the shortest the one with the fewest slices: 700
    // positions behind 12000 take 157 us in 220 slices and 159 to 171, for the same by these figures, in 244.)
    float low = limit, best_t = limit;
    int best_per = -1, best_parts = 0;
    for (;;) {
        int next = -1;
        for (int i = 0; i < tries; i++)
            if (least[i] >= 0.0f && (next < 0 || least[i] < least[next])) next = i;
        if (next < 0 || least[next] >= limit || least[next] >= 1.02f * low) break;
        least[next] = -1.0f;
        int parts;
        const float t = pf_time(b, c, pers[next], 1.02f * low, parts);
        if (t >= limit || t >= 1.02f * low) continue;
        low = t < low ? t : low;
        if (best_per < 0 || best_t >= 1.02f * low || parts < best_parts || (parts == best_parts && t < best_t))
            best_t = t, best_per = pers[next], best_parts = parts;
    }
    if (best_per < 0) return limit;
    best.per = best_per;
    best.first[0] = 0;
    for (int r = 0; r < b.count; r++)
        best.first[r + 1] = (uint16_t)(best.first[r] + (best_per ? pf_slices(b.tiles[r], b.plain[r], best_per) : 1));
    if (best.first[1] == 1) best.per = 0;   // (slices longer than any block)
    return best_t;
}

}  // namespace cwick
