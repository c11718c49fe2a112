// host_flags.hpp -- the numbers that kernels write to flags in host memory when a call's results are there, as the
// host counts them.  Plain C++.
#pragma once
#include <stdint.h>

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

}  // namespace cwick
