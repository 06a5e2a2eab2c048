// Rules of the launcher that look at sizes only: what a schedule holds for, how long the rows of a staged operand may become
// under it, which weights are read with the non-temporal hint, and where a plan is remembered. Host code.
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

// Whether the grouped GEMM reads `bytes` of weights (of the groups that have rows) with the non-temporal hint, which keeps the
// Infinity Cache (256 MiB, 268 MB) for other data. Measured without -> with it, us, on one set of weights (found in the cache as far as
// it holds them) and on sets in rotation:
//   strips of up to 256 columns: worth it once the cache no longer holds a part that counts. 2048 x 7168, 2 rows a group: 235 MB
//     45 -> 54, 57 -> 55; 264 MB 52 -> 60, 64 -> 60; 279 MB 56 -> 61, 65 -> 61; 294 MB 62 -> 62, 67 -> 63; 323 MB 68 -> 64, 69 -> 65; 396 MB
//     75 -> 68, 76 -> 69. 4096 x 2048, 20 rows: 243 MB 41 -> 48, 52 -> 49; 285 MB 65 -> 68, 72 -> 69; 302 MB 80 -> 72, 78 -> 72. Of 69 layouts
//     of 294 to 940 MB (all strips) none is more than 1 % slower with it; of 56 of 147 to 264 MB 37 are 10 to 36 % slower on weights that are in
//     the cache, which a caller that has just written them, or runs one layer again and again, has; in rotation those lose 1 to 12 % without it.
//   strips of 512 columns: 4096 x 2048, 2 rows: 260 MB 39 -> 42, 49 -> 43; 268 MB 41 -> 43, 50 -> 44; 277 MB 67 -> 64, 74 -> 69.
//   queue form: the tiles read activations again and again, which stay cached beside weights read with the hint, so it pays below the
//     cache's size too: 4096 x 2048, 300 rows a group on average, 218 MB 117 -> 107, 116 -> 115; 243 MB 121 -> 114, 122 -> 120; 7168 x 2048
//     250 MB 125 -> 113, 125 -> 126. Of 88 layouts of 190 to 940 MB one is 3 % slower in rotation (294 MB), the others by at most 1.4 %;
//     smaller ones not measured.
constexpr bool grouped_weights_streamed(double bytes, bool queue, int columns) {
    return bytes > (queue ? 192.0 * (1 << 20) : columns > 256 ? 256.0 * (1 << 20) : 290.0e6);
}

// Bits of the flags that a plan is chosen by (the launcher's kStageA and on).
constexpr int kStageBits = 9;

// Slot of a shape in the table of plans already worked out (a power of two of them, up to 2^25). All products unsigned: as an int the
// product of `stage`, of kStageBits, overflowed from 4 on.
constexpr unsigned plan_slot(int m, int n, int k, int stage, unsigned entries) {
    return ((((unsigned)m * 2654435761u) ^ ((unsigned)n * 2246822519u) ^ ((unsigned)k * 3266489917u) ^ ((unsigned)stage * 668265263u)) >> 7) % entries;
}

}  // namespace rf
