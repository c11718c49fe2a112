"""The rules that are plain C++ in headers of their own, compiled here for the CPU and checked over
their whole range: no GPU is involved."""
import os
import subprocess

from cwick_amd import build as B


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
