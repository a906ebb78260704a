// Arguments and launcher of the expert-grouped codebook GEMM (vq_gemm.hip):
// SwitchGLU's projections over VQ experts at prefill sizes.
#pragma once

#include "common.hpp"
#include "dispatch.hpp"

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
