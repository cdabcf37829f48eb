// mpm_radix_plan.hpp -- digits and scratch of the radix sort (host code only).
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <algorithm>

namespace mpm {

constexpr int SORT_TILE = 4096;  // keys per block
constexpr int MAX_DIGIT = 12;

constexpr uint32_t sort_blocks(uint32_t n) { return (n + SORT_TILE - 1) / SORT_TILE; }

// Digit width limit: the histogram table (2^width x blocks words, written and
// read once per pass) stays within 1 MB up to 512 blocks (2 M keys); beyond,
// 11 bits, because another pass over the keys costs more than the table.
inline int max_digit(uint32_t nb) {
    return nb <= 64 ? MAX_DIGIT : (nb <= 128 ? 11 : (nb <= 256 ? 10 : (nb <= 512 ? 9 : 11)));
}

struct RadixPlan {
    int passes, width;
};
inline RadixPlan radix_plan(uint32_t n, int bits) {
    const int w = max_digit(sort_blocks(n)), b = std::max(bits, 1);
    const int passes = (b + w - 1) / w;
    return {passes, (b + passes - 1) / passes};
}

// Words of the largest histogram table of any sort of up to nb blocks: the
// digits narrow as the blocks grow, so a table peaks at 64, 128, 256 and 512
// blocks, with the same 2^18 words each.
constexpr size_t table_words(uint32_t nb) {
    return nb <= 64 ? (size_t)nb << MAX_DIGIT : (nb <= 512 ? (size_t)1 << 18 : (size_t)nb << 11);
}

// Scratch of every sort of up to n keys, of any key width: the other half of
// the ping-pong keys and values, the histogram table, the digit totals.
constexpr size_t radix_scratch_words(uint32_t n) {
    return 2 * (size_t)n + table_words(sort_blocks(n)) + (1u << MAX_DIGIT) + 64;
}

}  // namespace mpm
