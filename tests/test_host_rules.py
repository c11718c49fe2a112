"""The rules that are plain C++ in headers of their own, compiled here for the CPU and checked over
their whole range: no GPU is involved."""
import os
import subprocess

from cwick_amd import build as B
from tests.test_gpu_dispatch_edges import PREFILL_ROUNDS


def run_cpp(tmp_path, header, body):
    """Compiles `body` (statements of main) behind `header` and runs it; what it prints comes back."""
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text("#define __host__\n#define __device__\n#include <cmath>\n#include <cstdio>\n#include <cstring>\n"
                   "#include <vector>\n#include <chrono>\n#include \"%s\"\nusing namespace cwick;\n%s\n"
                   % (os.path.join(B.CSRC, header), body))
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


def test_band_counters_follow_the_scores(tmp_path):
    """Every score is in one counter, the counters are in the order of the scores, a counter's range holds
    its scores and nothing of its neighbours', and the fine octaves have 128 counters each; for windows at
    both ends of the exponents and in between."""
    run_cpp(tmp_path, "band_counter.hpp", r"""
#define CHECK(x) do { if (!(x)) { printf("failed: %s, octave %u, bits %08x\n", #x, oct, bits); return 1; } } while (0)
int main() {
    for (uint32_t oct : {0u, 1u, 100u, 127u, 241u, 242u}) {
        uint32_t bits = 0, last = 0;
        float last_hi = -INFINITY;
        // all scores of twelve bits of fraction and the ones around them, from -inf to inf
        std::vector<float> v;
        for (uint32_t m = 0; m <= 0x7F800u; m++)
            for (int d = -1; d <= 1; d++) {
                const uint32_t b = (m << 12) + (uint32_t)d;
                float f;
                memcpy(&f, &b, 4);
                if (b <= 0x7F800000u && f == f) v.push_back(f);
            }
        const size_t half = v.size();
        std::vector<float> all;
        for (size_t i = half; i-- > 0;) all.push_back(-v[i]);
        all.insert(all.end(), v.begin(), v.end());
        for (float f : all) {
            memcpy(&bits, &f, 4);
            const uint32_t c = band_counter(f, oct);
            CHECK(c >= 1 && c < 4096);
            float lo, hi;
            band_range(c, oct, lo, hi);
            CHECK(f == 0.0f || (!(f < lo) && !(f > hi)));       // (a range that ends in a NaN is one the select refuses)
            CHECK(c >= last);
            if (c != last && last_hi == last_hi && lo == lo) CHECK(lo >= last_hi);
            const uint32_t e = bits >> 23 & 255;
            if (lo == lo && hi == hi && e >= oct && e < oct + BAND_OCTAVES && e > 0) CHECK(std::fabs(hi - lo) <= std::fabs(f) / 128);
            last = c;
            last_hi = hi;
        }
        CHECK(band_counter(NAN, oct) == 0 && band_counter(-NAN, oct) == 0);
        CHECK(band_counter(0.0f, oct) == band_counter(-0.0f, oct));
    }
    return 0;
}""")


def test_prefill_plan_is_near_the_best_and_quick(tmp_path):
    """The plan of a latent prefill chunk against all slice counts of all group sizes, by its own cost: at most
    3 % worse (the step between the counts it tries, a quarter, times the flatness of the optimum), and made in
    a fraction of the shortest kernel behind it.  5 us is several times what it takes here (about 1); trying
    every slice count took 24 for the last of the timed shapes and 38 for the longest."""
    out = run_cpp(tmp_path, "mla_plan.hpp", r"""
static float every_count(int64_t rb, int64_t tf, int64_t tl, int cus) {
    float best = 1e30f;
    for (int gsz = 4; gsz >= 1; gsz /= 2) {
        const int64_t g = (rb + gsz - 1) / gsz;
        if (gsz < 4 && g > cus) break;
        auto at = [&](int64_t i) { return (int)(tf + (tl - tf) * i / (g > 1 ? g - 1 : 1)); };
        auto whole = [&](int w) {
            float t = 0.0f;
            for (int d = 0; d < w; d += cus) t += plan_rounds(w - d < cus ? w - d : cus, at(g - 1 - d), plan_over(gsz), cus, 1.0f / cus);
            return t;
        };
        best = std::fmin(best, whole((int)g));
        const int full = (int)(g / cus * cus);
        for (int w = full; w >= 0 && w >= full - cus; w -= cus) {
            const int rest = (int)g - w, tiles = rest ? at(rest - 1) : 0;
            for (int s = 2; s <= tiles && rest && rest * s <= 4 * cus; s++)
                best = std::fmin(best, whole(w) + plan_sliced(gsz, rest, (tiles + s - 1) / s, s, cus, 1.0f / cus));
        }
    }
    return best;
}
int main() {
    float worst = 0.0f;
    for (int cus : {256, 64})
        for (int nhb : {1, 2, 3, 4, 6, 8})
            for (int64_t n = 1; n <= 3000; n = n < 40 ? n + 1 : n * 13 / 10)
                for (int64_t pos0 : {0, 100, 1291, 5000, 20000, 131072, 2000000}) {
                    const int64_t tf = (pos0 + 64) / 64, tl = (pos0 + n + 63) / 64;
                    const WidePlan p = plan_wide(n * nhb, tf, tl, cus);
                    const bool ok = (p.gsz == 1 || p.gsz == 2 || p.gsz == 4) && p.groups == (n * nhb + p.gsz - 1) / p.gsz &&
                                    p.whole <= p.groups && (p.whole == p.groups) == (p.slices == 1) &&
                                    (p.groups - p.whole) * p.slices <= 4 * (uint32_t)cus && (int64_t)p.slices <= tl;
                    if (!ok) { printf("bad plan: %d row blocks, %d at %d\n", (int)(n * nhb), (int)n, (int)pos0); return 1; }
                    if (p.groups > 16 * (uint32_t)cus) continue;
                    const float r = p.time / every_count(n * nhb, tf, tl, cus);
                    if (r > worst) worst = r;
                    if (r > 1.03f) { printf("%.3f: %d row blocks, %d at %d\n", r, (int)(n * nhb), (int)n, (int)pos0); return 1; }
                }
    double slowest = 0.0;
    for (int nhb : {1, 4, 8})
        for (int n : {1, 8}) {
            double best = 1e9;
            for (int rep = 0; rep < 20; rep++) {
                const auto t0 = std::chrono::steady_clock::now();
                volatile uint32_t sum = 0;
                for (int k = 0; k < 64; k++) sum = sum + plan_wide(n * nhb, 2047 + k, 2048 + k, 256).slices;
                const double us = std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count() / 64;
                if (us < best) best = us;
            }
            if (best > slowest) slowest = best;
        }
    printf("worst %.4f, slowest %.2f us\n", worst, slowest);
    return slowest < 5.0 ? 0 : 1;
}""")
    print(out)


def test_gqa_prefill_plan_of_one_round_of_blocks(tmp_path):
    """A chunk of exactly one round of whole blocks behind earlier keys is priced like its neighbours: no more than one
    of a position or a block more, and by both kernels."""
    print(run_cpp(tmp_path, "gqa_plan.hpp", r"""
int main() {
    for (int kv : {2, 4, 8})
        for (int rows : {64, 256}) {
            const PfCost &c = rows == 64 ? PF_COST_TEAM : PF_COST_WIDE;
            const int group = 16 / kv, P = rows / group, room = 256 / kv;
            for (int64_t pos0 : {1, 500, 2048, 4096, 8192, 16384})
                for (int64_t n : {(int64_t)room * P - P + 1, (int64_t)room * P}) {
                    PfPlan p;
                    const float t = pf_plan(pos0, n, P, kv, 0, 256, c, INFINITY, p);
                    for (int64_t more : {1, P}) {
                        const float u = pf_plan(pos0, room * P + more, P, kv, 0, 256, c, INFINITY, p);
                        if (t > 1.02f * u) { printf("%d kv heads, %d rows: %d at %d %.1f, %d %.1f\n", kv, rows, (int)n, (int)pos0, t, (int)(room * P + more), u); return 1; }
                    }
                }
        }
    return 0;
}"""))


def test_gqa_prefill_prices_follow_measured_plans(tmp_path):
    """The prices of plans that were timed (us): the faster of two has the lesser price, and none is a tenth off.  Two
    slices a block where the long ones lie on half of the XCDs; few units at work; the plan made of such a shape
    is within 5 % of the faster one (not all slice lengths are tried)."""
    print(run_cpp(tmp_path, "gqa_plan.hpp", r"""
struct Timed { int rows, per; float us; };
int main() {
    const struct { int64_t n, pos0; int heads, kv; Timed fast, slow; } shapes[] = {
        {2500, 4000, 16, 4, {256, 68, 251.4f}, {256, 152, 275.6f}}, {2500, 4000, 16, 2, {256, 59, 242.5f}, {256, 152, 270.7f}},
        {2800, 8000, 16, 4, {256, 0, 447.3f}, {256, 282, 480.9f}}, {2800, 8000, 16, 2, {256, 113, 446.1f}, {256, 282, 477.9f}},
        {3900, 6000, 8, 8, {256, 155, 267.4f}, {64, 0, 307.0f}}, {4000, 4000, 8, 8, {256, 125, 207.8f}, {64, 0, 237.6f}},
        {3700, 4000, 8, 8, {256, 121, 195.7f}, {64, 0, 213.4f}}, {1000, 16000, 8, 8, {256, 67, 138.5f}, {256, 66, 145.7f}},
    };
    for (auto &s : shapes) {
        static PfBlocks b[2];
        float t[2], best = INFINITY;
        for (int i = 0; i < 2; i++) {
            const Timed &p = i ? s.slow : s.fast;
            const int P = p.rows * s.kv / s.heads;
            b[i].count = (int)((s.n + P - 1) / P), b[i].n_kv_heads = s.kv, b[i].n_prec = 0, b[i].cus = 256;
            for (int r = 0; r < b[i].count; r++) {
                const int64_t pb = b[i].count - 1 - r;
                b[i].tiles[r] = (int)((pf_keys(s.pos0, s.n, P, pb) + PF_TK - 1) / PF_TK);
                b[i].plain[r] = (int)((s.pos0 + pb * P + 1) / PF_TK);
            }
            int parts;
            t[i] = pf_time(b[i], p.rows == 64 ? PF_COST_TEAM : PF_COST_WIDE, p.per, INFINITY, parts);
            if (std::fabs(t[i] / p.us - 1.0f) > 0.1f) { printf("%d behind %d: %d rows, %d tiles %.1f, took %.1f\n", (int)s.n, (int)s.pos0, p.rows, p.per, t[i], p.us); return 1; }
        }
        if (t[0] >= t[1]) { printf("%d behind %d of %d / %d: %.1f and %.1f\n", (int)s.n, (int)s.pos0, s.heads, s.kv, t[0], t[1]); return 1; }
        for (int rows : {64, 256}) {
            PfPlan p;
            const int P = rows * s.kv / s.heads;
            if ((s.n + P - 1) / P > PF_MAX_BLOCKS) continue;
            best = std::fmin(best, pf_plan(s.pos0, s.n, P, s.kv, 0, 256, rows == 64 ? PF_COST_TEAM : PF_COST_WIDE, INFINITY, p));
        }
        if (best > 1.05f * t[0]) { printf("%d behind %d of %d / %d: planned %.1f, there is %.1f\n", (int)s.n, (int)s.pos0, s.heads, s.kv, best, t[0]); return 1; }
    }
    return 0;
}"""))


def test_gqa_prefill_shapes_of_the_rounds_test(tmp_path):
    """What the plans make of the chunks that test_gqa_prefill_rounds runs: on 256 compute units the 64-row workgroups take
    them, and their steps are the ones that the test names."""
    out = run_cpp(tmp_path, "gqa_plan.hpp", r"""
int main() {
    static const int shapes[][4] = {SHAPES};
    for (auto &s : shapes) {
        const int n = s[0], pos0 = s[1], kv = s[3], group = s[2] / kv, rows[2] = {256 / group, 64 / group};
        int prec[2] = {0, 0}, blocks[2];
        static PfPlan wide, team;
        for (int k = 0; k < 2; k++) {
            blocks[k] = (n + rows[k] - 1) / rows[k];
            while (prec[k] < blocks[k] && pf_keys(pos0, n, rows[k], prec[k]) <= 1024) prec[k]++;
        }
        const float t = pf_plan(pos0, n, rows[0], kv, prec[0], 256, PF_COST_WIDE, INFINITY, wide);
        if (pf_plan(pos0, n, rows[1], kv, prec[1], 256, PF_COST_TEAM, t, team) >= t) { printf("%d at %d: not the 64-row workgroups\n", n, pos0); return 1; }
        unsigned steps[2] = {0, 0};
        for (int r = 0; r < blocks[1]; r++) {
            const int tiles = (int)(pf_keys(pos0, n, rows[1], blocks[1] - 1 - r) + PF_TK - 1) / PF_TK, cuts = team.first[r + 1] - team.first[r];
            for (int i = 0; i < cuts; i++) steps[blocks[1] - 1 - r < prec[1]] |= 1u << (((i + 1 < cuts ? team.per : tiles - i * team.per) + 3) / 4);
        }
        printf("%u %u\n", steps[0], steps[1]);
    }
}
""".replace("SHAPES", ", ".join("{%d, %d, %d, %d}" % shape for shape, _, _ in PREFILL_ROUNDS)))
    seen = [tuple([i for i in range(32) if int(w) >> i & 1] for w in line.split()) for line in out.splitlines()]
    assert seen == [(list(one), list(two)) for _, one, two in PREFILL_ROUNDS]


def test_gqa_prefill_plans_are_sound_and_quick(tmp_path):
    """The plans of both prefill kernels: the slices of every block cover its tiles, each begins below the
    diagonal and none is empty, there is room for the partials' numbers; less than a
    fifth behind the best of all slice lengths by its own cost (a dozen of them are tried, a quarter apart; here 17 %
    at the worst, where the other kernel's plan is a third shorter); a limit is kept; and a plan is made in a
    fraction of the kernel behind it: at most 10 us and an eighth of its time (on a loaded machine; here 1 us for
    200 positions, 5 for 1000, 11 for 4000, which take 160)."""
    out = run_cpp(tmp_path, "gqa_plan.hpp", r"""
int main() {
    float worst = 0.0f;
    const int cus = 256;
    for (int kv : {1, 2, 4, 8, 6})
            for (int rows : {64, 256})
                for (int group : {1, 4, 8})
                    for (int64_t n = 1; n <= 9000; n = n < 4 ? n + 1 : n * 17 / 10)
                        for (int64_t pos0 : {0, 31, 700, 5000, 16384, 1000000}) {
                            const PfCost &c = rows == 64 ? PF_COST_TEAM : PF_COST_WIDE;
                            const int P = rows / group;
                            const int64_t blocks = (n + P - 1) / P;
                            if (blocks > PF_MAX_BLOCKS) continue;
                            int64_t prec = 0;
                            while (prec < blocks && pf_keys(pos0, n, P, prec) <= 1024) prec++;
                            PfPlan p;
                            const float t = pf_plan(pos0, n, P, kv, prec, cus, c, INFINITY, p);
                            PfBlocks b;
                            b.count = (int)blocks, b.n_kv_heads = kv, b.n_prec = (int)prec, b.cus = cus;
                            bool ok = t > 0.0f && t < INFINITY && p.first[0] == 0;
                            for (int r = 0; r < b.count; r++) {
                                const int64_t pb = b.count - 1 - r;
                                b.tiles[r] = (int)((pf_keys(pos0, n, P, pb) + PF_TK - 1) / PF_TK);
                                b.plain[r] = (int)((pos0 + pb * P + 1) / PF_TK);
                                const int k = p.first[r + 1] - p.first[r];
                                ok = ok && k >= 1 && (p.per || k == 1);
                                ok = ok && (!p.per || p.first[b.count] * kv <= 4 * cus);       // the most that the header names
                                if (k > 1) ok = ok && (int64_t)(k - 1) * p.per < b.tiles[r] && (int64_t)(k - 1) * p.per * PF_TK <= pos0 + pb * P + 1;
                            }
                            if (!ok) { printf("bad plan: %d rows, %d at %d, %d kv heads of %d\n", rows, (int)n, (int)pos0, kv, group); return 1; }
                            PfPlan q;
                            if (pf_plan(pos0, n, P, kv, prec, cus, c, 0.5f * t, q) != 0.5f * t) { printf("limit not kept\n"); return 1; }
                            if (b.tiles[0] > 600 || (pos0 == 0 && b.count == cus / kv)) continue;      // (a prompt of one round stays whole)
                            int parts;
                            float best = pf_time(b, c, 0, INFINITY, parts);
                            for (int per = c.least; per < b.tiles[0]; per += c.waves) best = std::fmin(best, pf_time(b, c, per, best, parts));
                            if (t / best > worst) worst = t / best;
                            if (t > 1.2f * best) { printf("%.3f: %d rows, %d at %d, %d kv heads of %d, %d units\n", t / best, rows, (int)n, (int)pos0, kv, group, cus); return 1; }
                        }
    double slowest = 0.0;
    for (int64_t n : {16, 128, 360, 1000, 2500, 4000, 6000, 8000})
        for (int64_t pos0 : {0, 2000, 12000}) {
            double us = 1e9;
            float t = 0.0f;
            for (int rep = 0; rep < 20; rep++) {
                const auto t0 = std::chrono::steady_clock::now();
                PfPlan a, b;
                t = pf_plan(pos0, n, 64, 4, 0, 256, PF_COST_WIDE, INFINITY, a);
                if (n <= 8192) t = pf_plan(pos0, n, 16, 4, 0, 256, PF_COST_TEAM, t, b);
                us = std::fmin(us, std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count());
            }
            slowest = std::fmax(slowest, us / (10.0 + t / 8));
        }
    printf("worst %.3f, slowest %.2f of what it may take\n", worst, slowest);
    return slowest < 1.0 ? 0 : 1;
}""")
    print(out)


def test_flag_numbers_never_meet_an_old_flag(tmp_path):
    """Around the end of 32 bits: a call's number is never 0 (a flag never written) nor what any flag still holds,
    whether the calls before wrote all of their flags, some, or none."""
    run_cpp(tmp_path, "host_flags.hpp", r"""
int main() {
    for (uint32_t start : {0u, 0xFFFFFFF0u, 0xFFFFFFFEu, 0xFFFFFFFFu}) {
        uint32_t flags[8] = {0};
        FlagNumbers numbers;
        numbers.last = start;
        for (int i = 0; i < 8 && start; i++) flags[i] = i < 4 ? start : i - 3;     // old calls, and long ago the first ones
        for (int call = 0; call < 64; call++) {
            const uint32_t e = numbers.next(flags, 8);
            if (e == 0u) { printf("start %u call %d: number 0\n", start, call); return 1; }
            // (numbers of long ago: only once they run again)
            for (int i = 0; i < 8; i++)
                if (flags[i] == e) { printf("start %u call %d: flag %d holds %u\n", start, call, i, e); return 1; }
            for (int i = 0; i < call % 9; i++) flags[i] = e;
        }
    }
    return 0;
}""")


def test_watching_for_flags_ends(tmp_path):
    """Flags that arrive while they are watched are seen; where one does not arrive, the watch ends at its limit of
    half a millisecond (the best of five in less than two, on a loaded machine): no call keeps a core for longer."""
    run_cpp(tmp_path, "host_flags.hpp", r"""
int main() {
    using namespace std::chrono;
    uint32_t flags[4] = {7, 7, 7, 7};
    if (!flags_arrive(flags, 4, 7) || !flags_arrive(flags, 0, 9)) return 1;
    flags[3] = 6;
    double best = 1e9;
    for (int rep = 0; rep < 5; rep++) {
        const auto t0 = steady_clock::now();
        if (flags_arrive(flags, 4, 7)) return 2;
        const double us = duration<double, std::micro>(steady_clock::now() - t0).count();
        if (us < best) best = us;
    }
    printf("%.0f us\n", best);
    return best >= 500.0 && best < 2000.0 ? 0 : 3;
}""")


def test_mla_decode_slices(tmp_path):
    """The slices of an MLA decode: as many as the merge's test says; never more than the workspace is asked for, none
    empty; and by the rule's own figures never slower than a full round of workgroups."""
    from tests.test_gpu_dispatch_edges import MLA_SLICES
    cases = ", ".join("{%d, %d, %d, %d}" % c for c in MLA_SLICES)
    assert {s for _, _, _, s in MLA_SLICES} >= {2, 8, 9, 64, 65, 128, 129, 193, 256}
    run_cpp(tmp_path, "mla_plan.hpp", r"""
int main() {
    const int known[][4] = {CASES};
    for (auto &c : known) {
        const int64_t blocks = (c[1] + 31) / 32 * c[2], per = 64 * mla_decode_tiles((c[0] + 63) / 64, blocks, false, 1, 256);
        if ((c[0] + per - 1) / per != c[3]) { printf("%d keys of %d heads x %d: %d slices\n", c[0], c[1], c[2], (int)((c[0] + per - 1) / per)); return 1; }
    }
    for (int cus : {256, 304, 64})
        for (int per_cu : {1, 2, 8})
            for (bool list : {false, true})
                for (int64_t blocks : {1, 2, 3, 4, 8, 31, 32, 100, 256, 300, 16384})
                    for (int64_t tiles = 1; tiles < 40000000; tiles = tiles < 3000 ? tiles + 1 : tiles * 9 / 8) {
                        const int64_t per = mla_decode_tiles(tiles, blocks, list, per_cu, cus), most = mla_decode_most_splits(blocks, per_cu, cus);
                        const int64_t slices = (tiles + per - 1) / per, room = tiles < most ? tiles : most;
                        const int64_t full = (tiles + most - 1) / most, round = (tiles + full - 1) / full;
                        auto time = [&](int64_t t, int64_t n) { return (list ? 1.5 : 1.1) * t + (0.014 + 4e-5 * n * blocks) * n * blocks; };
                        if (per < 1 || slices < 1 || slices > room || slices > 1024 || (slices - 1) * per >= tiles ||
                            (per_cu == 1 && full <= 3 && tiles > 2 && time(per, slices) > time(full, round) * 1.0001)) {
                            printf("%d tiles, %d blocks, list %d, %d x %d: %d a slice, %d slices\n", (int)tiles, (int)blocks, list, per_cu, cus, (int)per, (int)slices);
                            return 1;
                        }
                    }
    return 0;
}""".replace("CASES", cases))
