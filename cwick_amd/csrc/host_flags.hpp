// host_flags.hpp -- the numbers that kernels write to flags in host memory when a call's results are there: how the
// host counts them, and how it watches for them.  Plain C++.
#pragma once
#include <stdint.h>

#include <chrono>

namespace cwick {

// One per piece of flags, so one per context: calls on a context follow each other, and a call ends when its
// flags are there (or its stream has been waited for).  A call's number is one that no flag of the piece holds:
// numbers go up from 1, and where they run out (after 2^32 - 1 calls, days of decoding) the flags are cleared,
// which nobody is writing between two calls, and the numbers start again.  The piece starts with flags of 0,
// which is no call's number.
struct FlagNumbers {
    uint32_t last = 0;
    uint32_t next(uint32_t *flags, int n) {
        if (++last == 0u) {
            for (int i = 0; i < n; i++) flags[i] = 0u;
            last = 1u;
        }
        return last;
    }
};

// All flags hold `number`; false when they do not within the limit, for which this keeps a core busy.  The calls
// that are watched take up to about 100 us (a decode over 128K keys); one that takes several times that,
// behind other work on the device, hands its core back and waits for the stream.
constexpr std::chrono::microseconds FLAG_WATCH{500};
inline bool flags_arrive(const uint32_t *flags, int count, uint32_t number) {
    const auto start = std::chrono::steady_clock::now();
    for (int i = 0, spins = 0; i < count;) {
        if (__atomic_load_n(flags + i, __ATOMIC_ACQUIRE) == number) {
            i++;
            continue;
        }
        __builtin_ia32_pause();
        if ((++spins & 127) == 0 && std::chrono::steady_clock::now() - start > FLAG_WATCH) return false;
    }
    return true;
}

}  // namespace cwick
