// Host-side rules of the prefill-shaped quantized matmul's launches: plain C++,
// so that they can be checked without a GPU.
#pragma once
#include <cstdint>

namespace eq {

// Whether a launch may read its scales and biases as whole words (two groups
// each): both arrays 4-byte aligned, rows of an even number of groups (always so
// below group size 64) and, with a split of K, splits that start at an even
// group.  A view at an odd element of a larger buffer is only 2-byte aligned;
// such a call reads its parameters two bytes at a time instead (4-bit group 32,
// 14336 x 4096: M = 512 80 us against 67 with windows, M = 64 28 against 23).
inline bool qmm_param_words(int gs, int K, int cps, const void* s, const void* b) {
    if ((reinterpret_cast<uintptr_t>(s) | reinterpret_cast<uintptr_t>(b)) % 4 != 0) return false;  // (no biases: null)
    return gs == 16 || gs == 32 || (gs == 64 && (K / 64) % 2 == 0 && cps % 2 == 0) ||
           (gs == 128 && (K / 128) % 2 == 0 && cps % 4 == 0);
}

}  // namespace eq
