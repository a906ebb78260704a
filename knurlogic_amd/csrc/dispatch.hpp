// Rules in sizes alone: which kernel a call takes and where a grid's
// workgroups go.  Plain C++ (no HIP), so the CPU tests compile it as it is.
#pragma once

#include <cstdint>

namespace kmi {

constexpr int64_t rule_ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// ---- the one-pass prompt attention's grid (sdpa_prefill.hip) -------------------
// units (a KV head's key split) x row tiles, the units ordered by unit % 8 and
// the whole cut into 8 runs of equal length, one per XCD (workgroup i runs on
// XCD i % 8).  From 8 units on, a unit's tiles share an XCD's L2; at any
// number no XCD is left with less.  (A whole unit per XCD left 4 of 8 idle at 4
// units: sdpa_prefill.hip has both sides.  Neighbouring units, the key splits
// of one head, on one XCD measured 3% slower at 16000 keys.)
constexpr int SP_XCDS = 8;

struct SpPlace {
    int unit, tile;         // unit -1: nothing to do
};

constexpr int sp_run(int units, int row_tiles) {
    return (int)rule_ceil_div((int64_t)units * row_tiles, SP_XCDS);
}

constexpr SpPlace sp_place(int id, int units, int row_tiles) {
    const int run = sp_run(units, row_tiles), at = id % SP_XCDS * run + id / SP_XCDS;
    if (id / SP_XCDS >= run || at >= units * row_tiles) return SpPlace{-1, 0};
    // the q-th unit of the order: those of residues below units % 8 are one more
    const int q = at / row_tiles, few = units / SP_XCDS, more = units % SP_XCDS, q0 = more * (few + 1);
    const int unit = q < q0 ? q % (few + 1) * SP_XCDS + q / (few + 1)
                            : (q - q0) % few * SP_XCDS + more + (q - q0) / few;
    return SpPlace{unit, at % row_tiles};
}

// ---- microscaled dense products past 64 rows (qmv.hip) -------------------------
// The batched kernel's 64 x 64 tiles where they are so few that the GEMM's
// larger ones stage most of a tile as padding and then split K in short runs:
// mxfp4, batched against GEMM: 65 rows x [64, 14336] 16.1 and 20.2 us, 128 x
// [256, 4096] 12.9 and 16.3, 65 x [1000, 4096] 14.4 and 16.3, 1000 x [64, 14336] 19.9
// and 22.0; but 1000 x [256, 2048] 16.5 and 15.6, 65 x [1000, 14336] 27.0 and 24.3,
// 300 x [1000, 2048] 20.3 and 17.7.  (K is not split below 1024; there the GEMM
// is one launch for two: 65 x [64, 512] 13.0 and 11.0.)
constexpr bool mx_batched_wanted(int64_t M, int64_t N, int64_t K) {
    const int64_t tiles = rule_ceil_div(M, 64) * rule_ceil_div(N, 64);
    return K >= 1024 && tiles <= 32 && tiles * (K / 64) <= 4000;
}

}  // namespace kmi
