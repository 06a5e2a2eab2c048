// Sizes a schedule holds for, and how wide the rows of a staged operand may become under it. Host code only.
#pragma once

namespace rf {

// The persistent schedules keep a load cursor's K position in 32-bit per-lane offsets: K * M and K * N stay below 2^32.
constexpr bool persistent_offsets_fit(int m, int n, int k) {
    return (unsigned long long)k * m < (1ull << 32) && (unsigned long long)k * n < (1ull << 32);
}

// Length of a staged operand's rows: `x`, a multiple of 16, becomes whole cache lines where that adds no tile of `tile` rows or
// columns and, under a persistent schedule, where its offsets still fit (`other` is the operand's counterpart: N for rows of A).
// Without the second condition a plan chosen for x = 2097104 at K = 2048 was launched with 2097152 rows and refused.
constexpr int staged_length(int x, int tile, int other, int k, bool persistent) {
    const long lines = (x + 127L) / 128 * 128;
    if (lines > 0x7fffffffL || (lines + tile - 1) / tile != ((long)x + tile - 1) / tile) return x;
    return persistent && !persistent_offsets_fit((int)lines, other, k) ? x : (int)lines;
}

}  // namespace rf
