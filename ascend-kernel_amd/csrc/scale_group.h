// Which scale row a 32-k step of the int4 container belongs to: step / (steps per scale group), by a multiplication.
// No HIP in here: the host works the divider out, the kernels apply it, and a CPU test checks it.
#pragma once
#include <cstdint>

namespace moe {

// floor(step / d) = floor(step * mul / 2^(31 + shift)) with mul = 2^(31 + shift) / d rounded up, 2^shift <= d < 2^(shift + 1).
// The rounding moves step / d up by less than step / 2^(31 + shift) < step / 2^30 / d, which is less than the 1 / d that
// separates it from the next integer for every step below 2^30: for every K that the ops take.  (2^31 or 2^32 in place of
// 2^(31 + shift) give the row behind the last one from K = 1485120 or 2108800 on, with one group over all of K.)
struct ScaleRowDivider {
    uint32_t mul, shift;
};

constexpr ScaleRowDivider scale_row_divider(int64_t K, int64_t scale_rows) {
    const uint64_t d = scale_rows > 0 && K / scale_rows >= 32 ? (uint64_t)(K / scale_rows) >> 5 : 1;
    uint32_t shift = 0;
    while (d >> (shift + 1)) ++shift;
    return {(uint32_t)(((uint64_t{1} << (31 + shift)) + d - 1) / d), shift};
}

constexpr uint32_t scale_row(ScaleRowDivider r, uint32_t step) { return (uint32_t)(((uint64_t)(2 * step) * r.mul) >> 32) >> r.shift; }

}  // namespace moe
