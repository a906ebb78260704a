// Rules in sizes alone: which kernel a call takes and where a grid's
// workgroups go.  Plain C++ (no HIP), so the CPU tests compile it as it is.
#pragma once

#include <cstdint>

namespace kmi {

constexpr int64_t rule_ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// ---- the one-pass prompt attention's grid (sdpa_prefill.hip) -------------------
// units (a KV head's key split) x row tiles.  Unit u whole on XCD u % 8
// (workgroup i runs on XCD i % 8), whose L2 then holds its K and V; where that
// gives some XCD more workgroups per CU than an even share would, the units
// ordered by u % 8 and the whole cut into 8 runs of equal length.  2048 queries over
// 4000 keys, whole units and cut, us: 32 heads over 4 KV heads, D = 128 435 and
// 229, 16 over 2, D = 256 1526 and 419; 300 x 3000, 16 over 2, D = 256 131 and 74.  Cut
// without that need it is slower: 96 queries over 3387 keys, 32 over 4, D = 128 (44
// units of 6 tiles: 36 workgroups on one XCD's 32 CUs, 33 if cut) 39 and 42.
constexpr int SP_XCDS = 8, SP_XCD_CUS = 32;

struct SpPlace {
    int unit, tile;         // unit -1: nothing to do
};

// workgroups on the fullest XCD: whole units, and cut
constexpr int sp_whole(int units, int row_tiles) { return (units + SP_XCDS - 1) / SP_XCDS * row_tiles; }
constexpr int sp_cut(int units, int row_tiles) {
    return (int)rule_ceil_div((int64_t)units * row_tiles, SP_XCDS);
}
constexpr bool sp_is_cut(int units, int row_tiles) {
    return (sp_whole(units, row_tiles) - 1) / SP_XCD_CUS > (sp_cut(units, row_tiles) - 1) / SP_XCD_CUS;
}
// the grid's workgroups per XCD
constexpr int sp_run(int units, int row_tiles) {
    return sp_is_cut(units, row_tiles) ? sp_cut(units, row_tiles) : sp_whole(units, row_tiles);
}

constexpr SpPlace sp_place(int id, int units, int row_tiles) {
    const int run = sp_run(units, row_tiles), xcd = id % SP_XCDS, at = id / SP_XCDS;
    if (at >= run) return SpPlace{-1, 0};
    if (!sp_is_cut(units, row_tiles)) {
        const int unit = SP_XCDS * (at / row_tiles) + xcd;
        return SpPlace{unit < units ? unit : -1, at % row_tiles};
    }
    if (xcd * run + at >= units * row_tiles) return SpPlace{-1, 0};
    // the q-th unit of the order: those of residues below units % 8 are one more
    const int q = (xcd * run + at) / row_tiles, few = units / SP_XCDS, more = units % SP_XCDS, q0 = more * (few + 1);
    const int unit = q < q0 ? q % (few + 1) * SP_XCDS + q / (few + 1)
                            : (q - q0) % few * SP_XCDS + more + (q - q0) / few;
    return SpPlace{unit, (xcd * run + at) % row_tiles};
}

// ---- microscaled dense products past 64 rows (qmv.hip) -------------------------
// The batched kernel's 64 x 64 tiles where they are so few that the GEMM's
// larger ones stage most of a tile as padding and then split K in short runs:
// mxfp4, batched against GEMM: 65 rows x [64, 14336] 16.1 and 20.2 us, 128 x
// [256, 4096] 12.9 and 16.3, 65 x [1000, 4096] 14.4 and 16.3, 1000 x [64, 14336] 19.9
// and 22.0; but 1000 x [256, 2048] 16.5 and 15.6, 65 x [1000, 14336] 27.0 and 24.3,
// 300 x [1000, 2048] 20.3 and 17.7.  At K = 1024 device time differs at twice the
// outputs too: 129 x [1000, 1024] 12.0 and 13.8, 1000 x [256, 1024] 13.1 and 14.1.  (K is
// not split below 1024; there the GEMM is one launch for two: 65 x [64, 512] 13.0
// and 11.0.)
constexpr bool mx_batched_wanted(int64_t M, int64_t N, int64_t K) {
    const int64_t tiles = rule_ceil_div(M, 64) * rule_ceil_div(N, 64);
    return K >= 1024 && tiles <= (K < 2048 ? 64 : 32) && tiles * (K / 64) <= 4000;
}

// ---- codebook experts: grouped GEMM or 16-row expert tiles (vq.hip, vq_packed.hip)
// 32-row blocks of the largest tile the grouped GEMM takes, and its rows
// (code_bytes 0: packed fields of vectors of dim)
constexpr int vqg_max_blocks(int code_bytes, int dim) { return code_bytes ? 5 : dim == 2 ? 2 : 4; }
constexpr int vqg_tile_rows(int code_bytes, int dim) { return 32 * vqg_max_blocks(code_bytes, dim); }

// Whether P routed pairs over E experts, avg rows per routed expert, H -> I -> H,
// run on the grouped GEMM (vq_gemm.hip) rather than on the 16-row expert tiles,
// whose time grows with the rows while the GEMM's is nearly flat up to 32 rows
// per expert.  The GEMM wants its gate/up grid to fill CUs (g: workgroups of a
// largest tile and 256 output columns, one per CU) and rows enough per tile, the
// fewer the more inputs share what a tile sets up; g, rows and H trade.  The
// lines come from 2018 calls timed on both, 4 to 128 experts, 1024..3072 -> 256..1536,
// 3 to 400 rows; none takes the kernel that was over 3% slower.  Nearest to them,
// 16-row tiles and GEMM, us:
//   one-byte codes: 128 experts 2048 -> 768 (g 384), 16 rows 112 and 103; 40 experts
//     (g 120), 47 rows 88 and 78; 32 experts (g 96), 32 rows 63 and 63; 1024 -> 512: 60
//     experts (g 120), 24 rows 47 and 48, 32 experts (g 64), 128 rows 74 and 85, 8 experts (g
//     16) 37 and 77; 1536 -> 1024: 128 experts, 16 rows 98 and 103, 96 experts, 30 rows
//     123 and 110.
//   16-bit codes (a tile stages its codebook, 64 KB at 4096 x 8): 128 experts 2048 ->
//     768, 3 rows 117 and 108; 48 experts 2048 -> 512 (g 96), 7 rows 69 and 52; 16 experts 2048
//     -> 768 (g 48), 32 rows 75 and 62; 8 experts (g 24), 128 rows 93 and 108; 1024 -> 512:
//     128 experts (g 256), 3 rows 44 and 49; 60 experts (g 120), 8 rows 41 and 43; 32 experts
//     (g 64), 16 rows 42 and 42, 32 rows 51 and 49; 16 experts (g 32), 32 rows 44 and 47.
//   packed vectors of 4 and 8 (11-bit x 4): 128 experts 2048 -> 768, 5 rows 185 and 160;
//     32 experts (g 96), 12 rows 84 and 70; 16 experts 2048 -> 512 (g 32), 24 rows 59 and 72;
//     1280 -> 512: 32 experts (g 64), 12 rows 50 and 56, 24 rows 63 and 60; 8 experts (g 16),
//     48 rows 45 and 58.
//   vectors of 8 (8-bit, one gather each) from fewer: 32 experts 3072 -> 512 (g 64),
//     23 rows 117 and 80; 24 experts 2048 -> 768 (g 72), 20 rows 82 and 63.
//   vectors of 2: 128 experts 2816 -> 704, 17 rows 388 and 363; 48 experts 3072 -> 512 (g
//     96), 22 rows 161 and 185; 24 experts 1024 -> 512 (g 48), 56 rows 67 and 75; 24
//     experts 2048 -> 512 (g 48), 54 rows 137 and 108.
constexpr bool vqg_wanted(int code_bytes, int dim, int64_t P, int64_t E, int64_t avg, int64_t H, int64_t I) {
    const int64_t blocks = vqg_max_blocks(code_bytes, dim), full = avg / (32 * blocks);
    const int64_t rest = rule_ceil_div(avg - full * 32 * blocks, 32);
    const int64_t g = (P < E ? P : E) * rule_ceil_div(I, 256) * (full ? full * blocks + rest : rest) /
                      (full ? blocks : rest ? rest : 1);
    const bool wide = H >= 2048;
    if (code_bytes == 2) {
        if (H >= 1536)
            return (wide && g >= 384 && avg >= 3) || (g >= 128 && avg >= 6) || (g >= 96 && avg >= 7) ||
                   (g >= 80 && avg >= 9) || (g >= 64 && avg >= 19) || (wide && g >= 48 && avg >= 32) ||
                   (g >= 38 && avg >= 120);
        return (g >= 128 && avg >= 10) || (g >= 80 && avg >= 24) || (g >= 64 && avg >= 38) || (g >= 48 && avg >= 140);
    }
    if (code_bytes == 1)
        return P >= 1024 && ((g >= 128 && avg >= (H >= 2 * I ? 16 : 24)) || (g >= 96 && avg >= (wide ? 40 : 64)) ||
                             (wide && g >= 72 && avg >= 200));
    if (dim == 2) return P >= 1024 && avg >= (g >= 120 ? 17 : 24) && (g >= 56 || (g >= 40 && (wide || avg >= 140)));
    if (P < 384 || avg < (P >= 640 ? 5 : 12)) return false;
    if (dim == 8 && ((g >= 80 && avg >= 12) || (g >= 64 && avg >= 20) || (wide && g >= 40 && avg >= 20) ||
                     (wide && g >= 24 && avg >= 100)))
        return true;
    return g >= 128 || (g >= 96 && avg >= (wide ? 12 : 16)) || (g >= 80 && avg >= 18) || (g >= 64 && avg >= 24) ||
           (g >= (wide ? 32 : 40) && avg >= 36) || (wide && g >= 27 && avg >= 140);
}

// ---- 4-bit experts from 64 rows each: moe_eg's tiles or moe_gemm's -------------
// Both run one workgroup per CU, so a projection takes rounds of the CUs.  A
// moe_gemm round is a whole tile (128 rows x 256 weight rows, or 256 x 128 past 128
// rows per expert) whatever it holds; moe_eg's workgroups take 512 weight rows and
// their time follows their 32-row blocks, each 0.36 of a moe_gemm round.  Wins
// where the experts' rows leave moe_gemm's tiles part empty or spill a few rows
// into a second tile; loses where one round of moe_gemm holds them all.
// moe_gemm and moe_eg, us: 128 experts 2048 -> 768, 64 rows 267 and 208, 128 rows
// 412 and 277; 48 experts 1024 -> 768, 64 rows 97 and 73; 32 experts 2048 -> 1024, 80
// rows 94 and 104, 128 rows 161 and 127; 16 experts 2048 -> 2048, 96 rows 106 and 124; 32
// experts 1536 -> 512, 170 rows 85 and 99, 256 rows 132 and 103; 32 experts 1024 ->
// 512, 166 rows 66 and 88, 317 rows 113 and 92.  Below half a grid (32 experts 1536
// -> 512, 64 rows: 70 and 79) moe_gemm stays.
constexpr int EG_MAX_BLOCKS = 5;             // row blocks of moe_eg's largest tile
constexpr int64_t EG_MIN_GRID = 128;

constexpr bool moe_eg_wanted(int64_t active, int64_t rows, int64_t H, int64_t I) {
    constexpr int64_t TILE = 32 * EG_MAX_BLOCKS, CUS = 256;
    if (active * rule_ceil_div(rows, TILE) * rule_ceil_div(I, 256) < EG_MIN_GRID) return false;
    int64_t dev = 0;                         // routed rows spread by about their root
    while ((dev + 1) * (dev + 1) <= rows) dev++;
    const int64_t most = rows + dev;
    const int64_t bm = rows <= 128 ? 128 : 256, tiles = active * rule_ceil_div(most, bm);
    const int64_t gemm = rule_ceil_div(tiles * rule_ceil_div(I, 16384 / bm), CUS) * H +
                         rule_ceil_div(tiles * rule_ceil_div(H, 32768 / bm), CUS) * I;
    // row blocks of an expert, and of its largest tile
    const int64_t full = most / TILE, rest = rule_ceil_div(most - full * TILE, 32);
    const int64_t blocks = EG_MAX_BLOCKS * full + rest, largest = full ? EG_MAX_BLOCKS : rest;
    const int64_t up = active * rule_ceil_div(I, 256) * blocks, down = active * rule_ceil_div(H, 512) * blocks;
    const int64_t eg = (up > largest * CUS ? up : largest * CUS) * H + (down > largest * CUS ? down : largest * CUS) * I;
    return 36 * eg < 100 * CUS * gemm;
}

}  // namespace kmi
