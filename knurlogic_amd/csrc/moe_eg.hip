// SwitchGLU's two projections over 4-bit affine experts at prefill sizes
// (src/knurlogic/engine/families/glm5/architecture/glm5_next/_mlx_vlm/models/
// switch_layers.py:71-86,172-193): rows grouped by expert (the GPU sort), one
// tile of up to 160 rows per workgroup and column block.
//
// The codebook GEMM's structure (vq_gemm.hip): the 8 waves split the columns
// only (64 weight rows each: 64 columns, or the gate and up rows of 32), so a
// wave dequantizes its own weights straight into v_mfma_f32_32x32x16_bf16's B
// operand -- no LDS pass, no barrier for B -- and every wave runs
// ceil(count / 32) row blocks, compiled per block count.  moe_gemm.hip's tiles
// are 128 or 256 rows whatever an expert sees: at 128 rows per expert on
// average half the experts take a second tile of a few rows at a full tile's
// cost.
//   - x rows (bf16) and packed codes arrive by direct-to-LDS loads, S - 1
//     stages of 64 inputs ahead, codes one stage earlier than x; a stage's wait
//     is a counted vmcnt (nothing else in the loop touches global memory).  The
//     expert's scales and biases for the wave's rows are loaded once.
//   - weights are bf16(s * q + b), one rounding, as moe_gemm's; the next MFMA
//     step's are formed between this step's MFMAs, piece by piece.
// Measured, 128 experts 2048 -> 768 -> 2048, top-8, 2048 tokens: gate/up 256 us on
// moe_gemm, 161 here, down 131 -> 87 (what is left over the matrix cores' time:
// 384 gate/up workgroups on 256 CUs, and the dequantization's vector
// instructions beside 8 MFMAs per row block).
#include "dispatch.hpp"
#include "qgemv.hpp"

namespace kmi {

namespace {

#define KMI_EG_LDS(p) ((__attribute__((address_space(3))) void*)(p))

__device__ __forceinline__ void eg_dma16(__amdgpu_buffer_rsrc_t r, unsigned char* lds, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, KMI_EG_LDS(lds), 16, voff, soff, 0, 0);
}

template <int N_>
__device__ __forceinline__ void eg_wait() {
    static_assert(N_ >= 0 && N_ < 64, "vmcnt");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N_) : "memory");
}

__device__ __forceinline__ f32x16 eg_mfma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(a), as_bf16x8(b), c, 0, 0, 0);
}

constexpr uint32_t EG_NONE = 0x80000000u;    // an offset past every view: reads 0
constexpr int EG_BK = 64, EG_WAVES = 8;
constexpr int EG_MAX_NB = EG_MAX_BLOCKS;
constexpr int EG_RIDS = 192;                 // tile rows staged (whole 64-row loads)
constexpr int EG_CODES = 2048;               // a wave's codes per stage: 64 rows of 32 bytes

constexpr int eg_a_bytes(int nb) { return (nb + 1) / 2 * 8192; }
constexpr int eg_stages(int nb) { return nb <= 2 ? 3 : 2; }
constexpr int eg_ring(int nb) { return eg_stages(nb) * (eg_a_bytes(nb) + EG_WAVES * EG_CODES); }
constexpr int eg_max_ring() {
    int m = 0;
    for (int nb = 1; nb <= EG_MAX_NB; nb++) m = eg_ring(nb) > m ? eg_ring(nb) : m;
    return m;
}
// a wave's scales or biases of 32 rows, in whole 1 KB loads: 16-byte pieces of
// 8 groups, piece-major (row l's at 16 l: a stage's reads of 32 rows fall on
// distinct banks; row-major they cost a fifth of the kernel)
__host__ __device__ constexpr int eg_sc_bytes(int G) { return ((G + 7) / 8 * 512 + 1023) / 1024 * 1024; }

template <int GS, bool GLU, int NB>
__device__ __forceinline__ void eg_body(const QgArgs& a, int expert, int nt, unsigned char* smem, const int32_t* rid_s) {
    constexpr int NA = (NB + 1) / 2, AB = eg_a_bytes(NB), S = eg_stages(NB), PER = NA + 2;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, h = lane >> 5;
    const int K = (int)a.K, nk = K / EG_BK, G = K / GS;
    const int scb = eg_sc_bytes(G);
    unsigned char* sw = smem + wave * (4 * scb);                 // this wave's scales / biases, rows of block 0 / 1
    unsigned char* ar = smem + EG_WAVES * 4 * scb;
    unsigned char* cr = ar + S * AB + wave * EG_CODES;           // this wave's codes

    const __amdgpu_buffer_rsrc_t rx = make_rsrc(a.x, a.xrows * a.K * 2);
    uint32_t xoff[NA];
#pragma unroll
    for (int j = 0; j < NA; j++) {
        const int m = 8 * (wave + 8 * j) + lane / 8, p = (lane % 8) ^ ((m >> 1) & 7);
        const int r = rid_s[m];
        const int64_t xr = r < 0 ? -1 : (int64_t)r / a.lhs_div;
        xoff[j] = xr >= 0 && xr < a.xrows ? (uint32_t)((xr * a.K + p * 8) * 2) : EG_NONE;
    }
    // block j's first weight row within the expert's view, and this lane's
    // output column; a row past the view reads zeros
    const int64_t wpr = a.K / 8, e0 = (int64_t)expert * a.erows;
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(a.w + e0 * wpr, a.erows * wpr * 4);
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(a.s + e0 * G, a.erows * G * 2);
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(a.b + e0 * G, a.erows * G * 2);
    int col[2];
    int64_t row0[2];
    uint32_t coff[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int c0 = GLU ? nt * 256 + 32 * wave : nt * 512 + 64 * wave + 32 * j;
        col[j] = c0 + l32;
        row0[j] = (GLU && j ? a.up_off : 0) + c0;
        const int64_t r = row0[j] + l32;
        coff[j] = r < a.erows ? (uint32_t)(r * wpr * 4 + 16 * h) : EG_NONE;
    }
    auto issue_x = [&](int t) {
        const uint32_t so = t < nk ? (uint32_t)t * (EG_BK * 2) : EG_NONE;
        unsigned char* dst = ar + (t % S) * AB;
#pragma unroll
        for (int j = 0; j < NA; j++) eg_dma16(rx, dst + (wave + 8 * j) * 1024, xoff[j], so);
    };
    auto issue_c = [&](int t) {
        const uint32_t so = t < nk ? (uint32_t)t * 32 : EG_NONE;
        unsigned char* dst = cr + (t % S) * (EG_WAVES * EG_CODES);
#pragma unroll
        for (int j = 0; j < 2; j++) eg_dma16(rw, dst + j * 1024, coff[j], so);
    };
    issue_c(0);
    // scales and biases of block j's 32 rows.  Rows of an odd number of groups
    // start between words, where 16-byte loads may not: their 32 rows are
    // loaded as they lie in memory
    const bool odd = G & 1;
    const int scrow = odd ? 2 * G : 16, scpiece = odd ? 16 : 512;
#pragma unroll
    for (int j = 0; j < 2; j++)
        for (int q = 0; q < scb; q += 1024) {
            const int u = q / 16 + lane;
            const int64_t off = row0[j] * G * 2 + (odd ? 16 * u : (u % 32) * G * 2 + (u / 32) * 16);
            const uint32_t v = row0[j] < a.erows ? (uint32_t)off : EG_NONE;
            eg_dma16(rs, sw + (2 * j) * scb + q, v, 0);
            eg_dma16(rb, sw + (2 * j + 1) * scb + q, v, 0);
        }
#pragma unroll
    for (int t = 0; t < S - 1; t++) {
        issue_x(t);
        issue_c(t + 1);
    }
    eg_wait<0>();
    lds_barrier();

    // a stage's codes, scale and bias of this lane's two weight rows
    struct Stage {
        u32x4 w[2];
        float s[2], b[2];
    };
    auto read_stage = [&](int t0) -> Stage {
        Stage c;
        const int t = t0 < nk ? t0 : nk - 1;
        const unsigned char* src = cr + (t0 % S) * (EG_WAVES * EG_CODES);
        const int g = GS == 128 ? t >> 1 : t;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            c.w[j] = *(const u32x4*)(src + j * 1024 + lane * 16);
            const unsigned char* p = sw + (2 * j) * scb + l32 * scrow + (g >> 3) * scpiece + (g & 7) * 2;
            c.s[j] = bf16_to_f32(*(const uint16_t*)p);
            c.b[j] = bf16_to_f32(*(const uint16_t*)(p + scb));
        }
        return c;
    };
    // weights 2 d, 2 d + 1 of block j's word, split into bytes
    uint32_t ev[2], od[2];
    auto split = [&](const Stage& c, int j, int s) { nibble_bytes(c.w[j][s], ev[j], od[j]); };
    auto piece = [&](const Stage& c, int j, int d) -> uint32_t {
        return cvt_pk_bf16(__builtin_fmaf(c.s[j], (float)((ev[j] >> (8 * d)) & 0xffu), c.b[j]),
                           __builtin_fmaf(c.s[j], (float)((od[j] >> (8 * d)) & 0xffu), c.b[j]));
    };
    // x fragment of row block i, step s: row 32 i + l32, piece 4 h + s
    uint32_t aoff[4];
#pragma unroll
    for (int s = 0; s < 4; s++)
        aoff[s] = (uint32_t)l32 * 128 + 16u * ((uint32_t)(4 * h + s) ^ ((uint32_t)(l32 >> 1) & 7u));
    auto read_x = [&](const unsigned char* base, int i, int s) -> u32x4 {
        return *(const u32x4*)(base + i * 4096 + aoff[s]);
    };

    f32x16 acc[NB][2];
#pragma unroll
    for (int i = 0; i < NB; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

    Stage cw = read_stage(0);
    u32x4 B[2][2];                                  // [step parity][block]
#pragma unroll
    for (int j = 0; j < 2; j++) {
        split(cw, j, 0);
#pragma unroll
        for (int d = 0; d < 4; d++) B[0][j][d] = piece(cw, j, d);
    }
    for (int t = 0; t < nk; t++) {
        eg_wait<PER*(S - 2)>();                     // this wave's x of stage t and codes of t + 1 are in LDS
        lds_barrier();                              // and every wave's x
        issue_x(t + S - 1);
        issue_c(t + S);
        const unsigned char* base = ar + (t % S) * AB;
        const Stage cn = read_stage(t + 1);
        // fragment q = s * NB + i, read D ahead of its MFMAs
        constexpr int Q = 4 * NB, D = 3;
        u32x4 A[4];
#pragma unroll
        for (int q = 0; q < D; q++) A[q % 4] = read_x(base, q % NB, q / NB);
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const int s = q / NB, i = q % NB, c = s & 1;
            if (q + D < Q) A[(q + D) % 4] = read_x(base, (q + D) % NB, (q + D) / NB);
            // the next step's weights: piece p (block p / 4, pair p % 4) after
            // MFMA p * 2 NB / 8 of this step
#pragma unroll
            for (int j = 0; j < 2; j++) {
                __builtin_amdgcn_sched_barrier(0);
                acc[i][j] = eg_mfma(A[q % 4], B[c][j], acc[i][j]);
#pragma unroll
                for (int p = 0; p < 8; p++)
                    if (p * 2 * NB / 8 == 2 * i + j) {
                        const Stage& from = s < 3 ? cw : cn;
                        if (p % 4 == 0) split(from, p / 4, (s + 1) % 4);
                        B[c ^ 1][p / 4][p % 4] = piece(from, p / 4, p % 4);
                    }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        cw = cn;
    }

    // D of block (i, j): tile row 32 i + 8 (r / 4) + 4 h + r % 4, this lane's
    // column of block j; through a buffer view of y, as moe_gemm's
    const __amdgpu_buffer_rsrc_t ry = make_rsrc(a.y, a.rows * a.N * 2);
    const uint32_t rowb = (uint32_t)a.N * 2;
    auto lo16 = [](uint32_t v) { return __uint_as_float(v << 16); };
    auto hi16 = [](uint32_t v) { return __uint_as_float(v & 0xffff0000u); };
#pragma unroll
    for (int i = 0; i < NB; i++) {
        int rid[16];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int4 v = *(const int4*)(rid_s + 32 * i + 8 * q + 4 * h);
            rid[4 * q] = v.x; rid[4 * q + 1] = v.y; rid[4 * q + 2] = v.z; rid[4 * q + 3] = v.w;
        }
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
#pragma unroll
            for (int j = 0; j < (GLU ? 1 : 2); j++) {
                uint32_t o;
                if constexpr (GLU) {
                    // act = round(round(silu_f32(round(gate))) * round(up))
                    const uint32_t g = cvt_pk_bf16(acc[i][0][r], acc[i][0][r + 1]);
                    const uint32_t u = cvt_pk_bf16(acc[i][1][r], acc[i][1][r + 1]);
                    o = cvt_pk_bf16(silu_bf16r(lo16(g)) * lo16(u), silu_bf16r(hi16(g)) * hi16(u));
                } else {
                    o = cvt_pk_bf16(acc[i][j][r], acc[i][j][r + 1]);
                }
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const uint32_t off = col[j] < a.N && rid[r + q] >= 0
                                             ? (uint32_t)rid[r + q] * rowb + (uint32_t)col[j] * 2 : EG_NONE;
                    __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(o >> (16 * q)), ry, (int)off, 0, 0);
                }
            }
        }
    }
    eg_wait<0>();                                   // no load still writes LDS when the workgroup ends
}

template <int GS, bool GLU>
__global__ __launch_bounds__(512, 1) void moe_eg_kernel(QgArgs a, int n_tiles, int tile_slots) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ __align__(16) int32_t rid_s[EG_RIDS];   // row id of tile row m (-1: none)
    // workgroup -> (tile, column block): the column blocks of a tile share an XCD
    const int id = (int)blockIdx.x, xcd = id & 7, kk = id >> 3;
    const int tile = 8 * (kk / n_tiles) + xcd, nt = kk % n_tiles;
    if (tile >= tile_slots) return;
    const int32_t* tp = a.tiles + 3 * (int64_t)tile;
    const int count = tp[2], expert = tp[0], start = tp[1];
    if (count <= 0 || count > 32 * EG_MAX_NB || expert < 0 || expert >= a.E) return;
    const int tid = threadIdx.x;
    if (tid < EG_RIDS) rid_s[tid] = tid < count ? a.sorted[start + tid] : -1;
    lds_barrier();
    const int nb = (count + 31) / 32;
    if (nb == 1) eg_body<GS, GLU, 1>(a, expert, nt, smem, rid_s);
    else if (nb == 2) eg_body<GS, GLU, 2>(a, expert, nt, smem, rid_s);
    else if (nb == 3) eg_body<GS, GLU, 3>(a, expert, nt, smem, rid_s);
    else if (nb == 4) eg_body<GS, GLU, 4>(a, expert, nt, smem, rid_s);
    else eg_body<GS, GLU, 5>(a, expert, nt, smem, rid_s);
}

size_t eg_lds(int64_t K, int gs) { return (size_t)EG_WAVES * 4 * eg_sc_bytes((int)(K / gs)) + eg_max_ring(); }

template <int GS>
int eg_go(const QgArgs& a, bool glu, int64_t tile_slots, hipStream_t st) {
    const size_t lds = eg_lds(a.K, GS);
    const int n_tiles = (int)ceil_div(a.N, glu ? 256 : 512);
    const int64_t wgs = 8 * n_tiles * ceil_div(tile_slots, 8);
    if (wgs >= (1LL << 31)) {
        set_error("moe_eg: grid of %lld workgroups", (long long)wgs);
        return EINVAL_ARG;
    }
    if (glu) {
        allow_dynamic_lds_once((const void*)moe_eg_kernel<GS, true>);
        moe_eg_kernel<GS, true><<<(unsigned)wgs, 512, lds, st>>>(a, n_tiles, (int)tile_slots);
    } else {
        allow_dynamic_lds_once((const void*)moe_eg_kernel<GS, false>);
        moe_eg_kernel<GS, false><<<(unsigned)wgs, 512, lds, st>>>(a, n_tiles, (int)tile_slots);
    }
    return OK;
}

}  // namespace

int moe_eg_tile_rows() { return 32 * EG_MAX_NB; }

bool moe_eg_supported(int64_t H, int64_t I, int bits, int gs, int mx) {
    return !mx && bits == 4 && (gs == 64 || gs == 128) && H % EG_BK == 0 && I % EG_BK == 0 && H % gs == 0 &&
           I % gs == 0 && eg_lds(H > I ? H : I, gs) + EG_RIDS * 4 <= 160 * 1024;
}

int launch_moe_eg(const QgArgs& a, int gs, bool glu, int64_t tile_slots, hipStream_t st) {
    if (!a.tiles || !a.sorted || a.mx || a.K % EG_BK || a.lhs_div < 1 || (glu && a.up_off <= 0) ||
        !moe_eg_supported(a.K, a.K, 4, gs, 0)) {
        set_error("moe_eg: expert tiles of 4-bit affine weights, groups of 64 or 128");
        return EINVAL_ARG;
    }
    if (!moe_eg_aligned(a.x, a.w, a.s, a.b)) {
        set_error("moe_eg: x and weights on 16 bytes, scales and biases on 4");
        return EINVAL_ARG;
    }
    if (a.xrows * a.K * 2 >= (1LL << 31) || a.erows * (a.K / 2) >= (1LL << 31) || a.rows * a.N * 2 >= (1LL << 31)) {
        set_error("moe_eg: x, y or an expert's weights past 2 GiB");
        return EINVAL_ARG;
    }
    return gs == 64 ? eg_go<64>(a, glu, tile_slots, st) : eg_go<128>(a, glu, tile_slots, st);
}

}  // namespace kmi
