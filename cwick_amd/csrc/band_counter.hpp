// band_counter.hpp -- the counters of the banded select's approximate scores: what the approximate kernel
// counts in and the classify kernel finds the threshold by.  Plain C++ but for the two qualifiers.
#pragma once
#include <stdint.h>

namespace cwick {

// The counter of a score among the 4096 of a row of the banded select: 0 for a NaN, otherwise counters in the
// order of the scores, two thousand for either sign.  The fourteen octaves from 2^(octave - 127) up have
// 128 counters each (seven bits of fraction), every other octave has one: the octaves that a row's largest
// scores can be in take most of the counters, and no score is without one.
constexpr uint32_t BAND_OCTAVES = 14;
constexpr int BAND_ABOVE = (int)BAND_OCTAVES * 127;          // number of an octave above those: its exponent and this
__host__ __device__ inline uint32_t band_counter(float f, uint32_t octave) {
    const uint32_t u = __builtin_bit_cast(uint32_t, f), mag = u & 0x7FFFFFFFu;
    const int e = (int)(mag >> 23), in = (int)octave + (int)(mag >> 16) - (int)(octave << 7);
    const int above = e + BAND_ABOVE, top = in < above ? in : above, m = e > top ? e : top;
    if (f != f) return 0u;
    return (uint32_t)(f < 0.0f ? 2047 - m : 2048 + m);
}
// the smallest and the largest score of a counter (not of 0)
__host__ __device__ inline void band_range(uint32_t counter, uint32_t octave, float &lo, float &hi) {
    const bool neg = counter < 2048u;
    const uint32_t m = neg ? 2047u - counter : counter - 2048u;
    uint32_t small, large;                                    // magnitudes
    if (m >= octave && m < octave + 128u * BAND_OCTAVES) {
        small = ((octave << 7) + (m - octave)) << 16;
        large = small | 0xFFFFu;
    } else {
        small = (m < octave ? m : m - (uint32_t)BAND_ABOVE) << 23;
        large = small | 0x7FFFFFu;
    }
    lo = __builtin_bit_cast(float, neg ? large | 0x80000000u : small);
    hi = __builtin_bit_cast(float, neg ? small | 0x80000000u : large);
}

}  // namespace cwick
