// Arguments and launcher of the expert-grouped codebook GEMM (vq_gemm.hip):
// SwitchGLU's projections over VQ experts at prefill sizes.
#pragma once

#include "common.hpp"

namespace kmi {

struct VqgArgs {
    const uint16_t* x;          // fp16 [xrows, K]
    int64_t xrows;
    int lhs_div;                // x row = row id / lhs_div
    const int32_t* tiles;       // the sort's [slots][3] (expert, start, count <= tile_rows)
    const int32_t* sorted;      // row ids grouped by expert
    int64_t E;
    const void* codes[2];       // [E, N, W]: one-byte, 16-bit or packed codes (set 1: the up rows)
    const uint16_t* sc[2];      // fp16 [E, N], packed: [E, N, K / group]
    const uint16_t* cb[2];      // fp16 [kc, 8], packed: [kc, dim]
    int kc;
    int64_t N, K;               // output columns (GLU: of act), inputs
    int64_t W;                  // packed: 32-bit words per row
    int group;                  // packed: inputs per scale
    uint16_t* y;                // [rows, N] bf16, or with y_f16 the same values as fp16
    int64_t rows;
    int y_f16;
};

// 32-row blocks of the largest tile the kernel takes, and its rows
constexpr int vqg_max_blocks(int code_bytes, int dim) { return code_bytes ? 5 : dim == 2 ? 2 : 4; }
constexpr int vqg_tile_rows(int code_bytes, int dim) { return 32 * vqg_max_blocks(code_bytes, dim); }

// Whether P routed pairs, avg rows per routed expert, run on this kernel
// rather than on the 16-row expert tiles, whose time grows with the rows
// while this kernel's is nearly flat up to 32 rows per expert.  Measured
// (16-row tiles against this kernel, us, 128 experts 2048 -> 768 -> 2048, top-8): one-byte
// codes 160 tokens (10 rows) 88 vs 103 us, 256 (16 rows) 111 vs 106; 16-bit
// codes (64 KB of codebook staged per tile) 33 tokens (3 rows) 114 vs 104,
// 100 tokens 133 vs 113; packed vectors of 4 64 tokens (4 rows) 150 vs 159, 80
// tokens (5 rows) 183 vs 167, 96 tokens 190 vs 160.  With 32 experts the few
// workgroups leave CUs idle and the lines lie higher: 640 pairs in one-byte
// codes (20 rows) 37 vs 48, packed 256 pairs (8 rows) 70 vs 70, 384 pairs (12
// rows) 83 vs 71; 40 experts 480 pairs (12 rows) 101 vs 73.  Vectors of 2 (four
// gathers per 8 inputs; 2816 -> 704): 100 experts 1600 pairs (16 rows) 322 vs
// 329, 1680 (17 rows) 330 vs 331, 128 experts 2048 pairs 388 vs 363; 64 experts
// 1026 pairs (17 rows) 210 vs 204; 32 experts 768 pairs (24 rows) 152 vs 164,
// 1024 (32 rows) 193 vs 167.
inline bool vqg_wanted(int code_bytes, int dim, int64_t P, int64_t avg) {
    if (code_bytes == 2) return avg >= 3;
    if (code_bytes == 1) return avg >= 16 && P >= 1024;
    if (dim == 2) return avg >= 17 && P >= 1024;
    return avg >= (P >= 640 ? 5 : 12) && P >= 384;
}

// whether the kernel covers a projection (code_bytes 1 or 2: per-channel
// scales, vectors of 8; 0: packed fields)
bool vqg_supported(int code_bytes, int pack_bits, int dim, int group, int64_t E, int64_t N, int64_t K, int kc,
                   bool two_cb);
// tile_slots: tiles of the sort (cut at vqg_tile_rows)
int launch_vqg(const VqgArgs& a, int code_bytes, int pack_bits, int dim, bool glu, int64_t tile_slots,
               hipStream_t st);
// bf16 [n] -> fp16 [n] (n a multiple of 8, both 16-byte aligned)
int launch_vqg_to_f16(const void* x, int64_t n, uint16_t* out, hipStream_t st);

}  // namespace kmi
