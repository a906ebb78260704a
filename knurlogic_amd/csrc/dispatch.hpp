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

}  // namespace kmi
