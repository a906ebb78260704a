// Codebook experts at prefill sizes (SwitchGLU over an artifact's
// VQSwitchLinear, src/knurlogic/engine/families/deepseek/heads/
// deepseek_v4.py:95-129): rows grouped by expert (the GPU sort), one tile of
// up to 160 rows per workgroup and column block, so a code is gathered once
// for all of its expert's rows.  The 16-row tiles of vq_mfma.hip gather an
// expert's codes once per 16 rows, which bounds them at prefill sizes.
//
//   - v_mfma_f32_32x32x16_f16: lane (n = l % 32, h = l / 32) of B is 8 inputs
//     of weight row n, i.e. one 8-element codebook vector, read from the LDS
//     codebook straight into the operand.  In a stage of 64 inputs lane half
//     h owns inputs [32 h, 32 h + 32), MFMA step s the 8 inputs at 32 h + 8 s,
//     for x and the weights alike.
//   - The 8 waves split the columns only (64 weight rows each: 64 columns, or
//     the gate and up rows of 32 columns), so no wave gathers another's
//     vectors and B never passes through LDS; every wave does the same
//     number of MFMAs, ceil(count / 32) row blocks (the body is compiled per
//     row-block count).
//   - x rows (fp16) and the raw codes arrive by direct-to-LDS loads, S - 1
//     stages ahead, one barrier per stage.  A stage's wait is a counted vmcnt:
//     nothing else in the loop touches global memory.  Codes are read by the
//     wave that loaded them (no barrier), one stage ahead of x, so a stage's
//     first gathers are in flight before its barrier.
//   - x row m keeps its 16-byte piece p at slot p ^ ((m / 2) % 8): 16 lanes'
//     reads of 16 consecutive rows fall on distinct bank groups.
// Packed fields carry a scale per group of 64 or 128 inputs: a stage's sum
// starts at zero and is multiplied by its scale in fp32 (as vq_packed_mfma
// does); one scale per channel multiplies the whole sum at the end.  Results
// are rounded as the other VQ kernels round (bf16 per projection, then the
// SwiGLU's two roundings).
// Measured, 128 experts 2048 -> 768 -> 2048, top-8: 4096 x 8 codebook, 2048
// tokens 934 us on the 16-row tiles, 257 here (gate/up 151, down 79 us: 384
// gate/up workgroups fill 256 CUs one and a half times); packed 2048 x 4, 512
// tokens 545 -> 179 (gate/up 109, down 53: the address units serve one weight
// row per lane).
#include "vq_gemm.hpp"

#include <type_traits>

namespace kmi {

namespace {

typedef _Float16 vqg_f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 vqg_f16x2 __attribute__((ext_vector_type(2)));

#define KMI_VQG_LDS(p) ((__attribute__((address_space(3))) void*)(p))

__device__ __forceinline__ f32x16 vqg_mfma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(vqg_f16x8, a), __builtin_bit_cast(vqg_f16x8, b),
                                                  c, 0, 0, 0);
}

// Direct-to-LDS loads: lane i's bytes land at lds + i * size.
__device__ __forceinline__ void vqg_dma16(__amdgpu_buffer_rsrc_t r, unsigned char* lds, uint32_t voff,
                                          uint32_t soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, KMI_VQG_LDS(lds), 16, voff, soff, 0, 0);
}
__device__ __forceinline__ void vqg_dma4(__amdgpu_buffer_rsrc_t r, unsigned char* lds, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, KMI_VQG_LDS(lds), 4, voff, soff, 0, 0);
}

// the same from each lane's own address
__device__ __forceinline__ void vqg_dma16_at(const void* p, unsigned char* lds) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)p, KMI_VQG_LDS(lds), 16, 0, 0);
}

template <int N_>
__device__ __forceinline__ void vqg_wait() {
    static_assert(N_ >= 0 && N_ < 64, "vmcnt");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N_) : "memory");
}

constexpr uint32_t VQG_NONE = 0x80000000u;   // an offset past every view: reads 0
constexpr int VQG_BK = 64;                    // inputs per stage
constexpr int VQG_WAVES = 8;
constexpr int VQG_RIDS = 192;                 // tile rows staged (whole 64-row loads)

// How a weight row's codes are laid out.  CB: bytes per code (1, 2), 0: PB-bit
// fields of vectors of DIM inputs.
template <int CB, int PB, int DIM>
struct VqgFmt {
    static constexpr bool PACKED = CB == 0;
    static constexpr int FPL = 32 / DIM;                     // codes of a lane per stage
    static constexpr int RUN = FPL * PB;                      // packed: their bits
    // packed: 16-byte loads that hold a run starting at any bit of a word
    // (16-bit fields start on a word)
    static constexpr int RL = PACKED ? (RUN + (PB == 16 ? 0 : 31) + 127) / 128 : 0;
    // direct-to-LDS loads of a wave per stage, and the LDS they fill: one-byte
    // codes 4 bytes per (row, half), 16-bit codes 16 bytes per row (two halves),
    // packed RL x 16 bytes per (row, half)
    static constexpr int LOADS = CB == 1 ? 2 : CB == 2 ? 1 : 2 * RL;
    static constexpr int BYTES = CB == 1 ? 512 : CB == 2 ? 1024 : 2 * RL * 1024;
    // stages in the ring by row blocks: as deep as the codebooks leave LDS for
    static constexpr int stages(int nb) {
        if (CB == 1) return nb <= 4 ? 4 : 3;
        if (CB == 2) return nb <= 2 ? 4 : nb <= 4 ? 3 : 2;
        return DIM == 2 || nb > 2 ? 2 : 3;
    }
    // gathers a whole stage ahead, into a second operand set, where the
    // registers allow it
    static constexpr bool ahead(int nb) { return stages(nb) >= 3 && nb <= (PACKED ? 2 : 4); }
    static constexpr int a_bytes(int nb) { return (nb + 1) / 2 * 8192; }
    static constexpr int ring(int nb) { return stages(nb) * (a_bytes(nb) + VQG_WAVES * BYTES); }
    // row blocks of the largest tile: as many as the registers hold (packed
    // fields need some for their group sums)
    static constexpr int MAX_NB = vqg_max_blocks(CB, DIM);
    static constexpr int max_ring() {
        int m = 0;
        for (int nb = 1; nb <= MAX_NB; nb++) m = ring(nb) > m ? ring(nb) : m;
        return m;
    }
};

// Packed: a wave's scales of 32 rows (two blocks of them), loaded once in whole
// 1 KB loads: 16-byte pieces of 8 groups, piece-major (row l's at 16 l), so a
// stage's reads of 32 rows fall on distinct banks
__host__ __device__ constexpr int vqg_sc_bytes(int G) { return ((G + 7) / 8 * 512 + 1023) / 1024 * 1024; }

struct VqgTile {
    int expert, count, nt;
};

template <class F, int CB, int PB, int DIM, bool GLU, int NB>
__device__ __forceinline__ void vqg_body(const VqgArgs& a, const VqgTile& tl, unsigned char* smem, const int32_t* rid_s,
                                         int cbstride, bool two_cb) {
    constexpr int NA = (NB + 1) / 2;               // x loads of a wave per stage
    constexpr int AB = F::a_bytes(NB);
    constexpr int S = F::stages(NB);
    constexpr int PER = NA + F::LOADS;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, h = lane >> 5;
    const int K = (int)a.K, nk = K / VQG_BK;
    const int G = F::PACKED ? K / a.group : 0;
    const int scb = F::PACKED ? vqg_sc_bytes(G) : 0;
    unsigned char* sw = smem + cbstride * (two_cb ? 2 : 1);
    unsigned char* ar = sw + VQG_WAVES * 2 * scb;
    sw += wave * 2 * scb;                                    // this wave's scales
    unsigned char* cr = ar + S * AB + wave * F::BYTES;       // this wave's codes, S slots apart by 8 waves

    // x: load j of wave w fills rows 8 (w + 8 j) .. + 7
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(a.x, a.xrows * a.K * 2);
    uint32_t xoff[NA];
#pragma unroll
    for (int j = 0; j < NA; j++) {
        const int m = 8 * (wave + 8 * j) + lane / 8, p = (lane % 8) ^ ((m >> 1) & 7);
        const int r = rid_s[m];
        const int64_t xr = r < 0 ? -1 : (int64_t)r / a.lhs_div;
        xoff[j] = xr >= 0 && xr < a.xrows ? (uint32_t)((xr * a.K + p * 8) * 2) : VQG_NONE;
    }
    // this lane's weight rows: block j (GLU: gate and up of one column)
    int col[2];
#pragma unroll
    for (int j = 0; j < 2; j++)
        col[j] = GLU ? tl.nt * 256 + 32 * wave + l32 : tl.nt * 512 + 64 * wave + 32 * j + l32;
    const int64_t e0 = (int64_t)tl.expert * a.N;
    const int gshift = F::PACKED && a.group == 128 ? 1 : 0;
    __amdgpu_buffer_rsrc_t rc[2];
    uint32_t coff[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int s = GLU ? j : 0;
        const int64_t rb = F::PACKED ? a.W * 4 : (int64_t)K / 8 * CB;    // bytes of a row's codes
        rc[j] = make_rsrc((const char*)a.codes[s] + e0 * rb, a.N * rb);
        const int n = col[j] < a.N ? col[j] : (int)a.N - 1;              // past N: a real row, never stored
        if constexpr (CB == 1) coff[j] = (uint32_t)(n * rb) + 4u * h;
        else coff[j] = (uint32_t)(n * a.W);                              // in words
        if constexpr (CB == 2) coff[j] = 0;
    }
    // 16-bit codes: lane r moves the 16 bytes (both halves) of the wave's row r
    const unsigned char* cptr = nullptr;
    if constexpr (CB == 2) {
        const int n0 = GLU ? tl.nt * 256 + 32 * wave + l32 : tl.nt * 512 + 64 * wave + lane;
        const int n = n0 < a.N ? n0 : (int)a.N - 1;
        cptr = (const unsigned char*)a.codes[GLU ? h : 0] + (e0 + n) * ((int64_t)K / 4);
    }
    // packed: the bit of this lane's first field of stage t within its row
    auto run_bit = [&](int t) -> uint32_t {
        return (uint32_t)((t * VQG_BK + 32 * h) / (F::PACKED ? DIM : 8)) * (uint32_t)PB;
    };

    auto issue_x = [&](int t) {
        const uint32_t so = t < nk ? (uint32_t)t * (VQG_BK * 2) : VQG_NONE;
        unsigned char* dst = ar + (t % S) * AB;
#pragma unroll
        for (int j = 0; j < NA; j++) vqg_dma16(rx, dst + (wave + 8 * j) * 1024, xoff[j], so);
    };
    auto issue_c = [&](int t0) {
        const int t = t0 < nk ? t0 : nk - 1;                             // past the last: its codes again, unused
        unsigned char* dst = cr + (t0 % S) * (VQG_WAVES * F::BYTES);
        if constexpr (CB == 1) {
#pragma unroll
            for (int j = 0; j < 2; j++) vqg_dma4(rc[j], dst + j * 256, coff[j], (uint32_t)t * 8);
        } else if constexpr (CB == 2) {
            vqg_dma16_at(cptr + t * 16, dst);
        } else {
            const uint32_t w0 = run_bit(t) >> 5;
#pragma unroll
            for (int j = 0; j < 2; j++) {
#pragma unroll
                for (int q = 0; q < F::RL; q++)
                    vqg_dma16(rc[j], dst + (j * F::RL + q) * 1024, (coff[j] + w0 + 4u * q) * 4u, 0);
            }
        }
    };

    issue_c(0);
    // Rows of an odd number of groups start between words, where 16-byte loads
    // may not: their 32 rows are loaded as they lie in memory
    const bool odd = G & 1;
    const int scrow = odd ? 2 * G : 16, scpiece = odd ? 16 : 512;
    if constexpr (F::PACKED) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const __amdgpu_buffer_rsrc_t rs = make_rsrc(a.sc[GLU ? j : 0] + e0 * G, a.N * G * 2);
            const int64_t row0 = col[j] - l32;
            for (int q = 0; q < scb; q += 1024) {
                const int u = q / 16 + lane;
                const int64_t off = row0 * G * 2 + (odd ? 16 * u : (u % 32) * G * 2 + (u / 32) * 16);
                vqg_dma16(rs, sw + j * scb + q, row0 < a.N ? (uint32_t)off : VQG_NONE, 0);
            }
        }
    }
#pragma unroll
    for (int t = 0; t < S - 1; t++) {
        issue_x(t);
        issue_c(t + 1);
    }
    // codebook(s) -> LDS through registers
    {
        const int cbytes = a.kc * (F::PACKED ? DIM : 8) * 2, pieces = cbytes / 16, tail = cbytes - pieces * 16;
        for (int s = 0; s < (two_cb ? 2 : 1); s++) {
            const __amdgpu_buffer_rsrc_t rcb = make_rsrc(a.cb[s], cbytes);
            unsigned char* dst = smem + s * cbstride;
            for (int p0 = tid; p0 < pieces; p0 += 512 * 8) {
                u32x4 v[8];
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    const int p = p0 + 512 * u;
                    v[u] = __builtin_amdgcn_raw_buffer_load_b128(rcb, p < pieces ? p * 16 : (int)VQG_NONE, 0, 0);
                }
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    const int p = p0 + 512 * u;
                    if (p < pieces) *(u32x4*)(dst + p * 16) = v[u];
                }
            }
            if (tid < tail / 4)
                *(uint32_t*)(dst + pieces * 16 + tid * 4) =
                    __builtin_amdgcn_raw_buffer_load_b32(rcb, pieces * 16 + tid * 4, 0, 0);
        }
    }
    vqg_wait<0>();
    lds_barrier();

    const uint32_t kcm1 = (uint32_t)(a.kc - 1);
    const unsigned char* cbl[2] = {smem, smem + (two_cb && GLU ? cbstride : 0)};
    // a stage's codes of this lane
    struct Codes {
        uint32_t w[2][F::PACKED ? 4 * F::RL : CB];
        uint32_t sc[2];
    };
    auto read_codes = [&](int t) -> Codes {
        Codes c = {};
        const int g = (t < nk ? t : nk - 1) >> gshift;
        const unsigned char* src = cr + (t % S) * (VQG_WAVES * F::BYTES);
#pragma unroll
        for (int j = 0; j < 2; j++) {
            if constexpr (CB == 1) c.w[j][0] = *(const uint32_t*)(src + j * 256 + lane * 4);
            else if constexpr (CB == 2) {
                const u32x2 v = *(const u32x2*)(src + (32 * j + l32) * 16 + 8 * h);
                c.w[j][0] = v.x; c.w[j][1] = v.y;
            } else {
#pragma unroll
                for (int q = 0; q < F::RL; q++) {
                    const u32x4 v = *(const u32x4*)(src + (j * F::RL + q) * 1024 + lane * 16);
                    c.w[j][4 * q] = v.x; c.w[j][4 * q + 1] = v.y; c.w[j][4 * q + 2] = v.z; c.w[j][4 * q + 3] = v.w;
                }
                c.sc[j] = *(const uint16_t*)(sw + j * scb + l32 * scrow + (g >> 3) * scpiece + (g & 7) * 2);
            }
        }
        return c;
    };
    // packed: bring a run to bit 0
    auto settle = [&](Codes& c, int t0) {
        if constexpr (F::PACKED) {
            const int t = t0 < nk ? t0 : nk - 1;
            const uint32_t sh = run_bit(t) & 31u;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                if constexpr (PB != 16) {
#pragma unroll
                    for (int q = 0; q < 4 * F::RL - 1; q++)
                        c.w[j][q] = __builtin_amdgcn_alignbit(c.w[j][q + 1], c.w[j][q], sh);
                }
            }
        }
    };
    // the codebook vector(s) of step s, row block j: 8 inputs
    auto gather = [&](const Codes& c, int j, int s) -> u32x4 {
        const unsigned char* cb = cbl[j];
        if constexpr (!F::PACKED) {
            uint32_t code;
            if constexpr (CB == 1) code = (c.w[j][0] >> (8 * s)) & 0xffu;
            else code = (c.w[j][s >> 1] >> (16 * (s & 1))) & 0xffffu;
            code = __builtin_elementwise_min(code, kcm1);
            return *(const u32x4*)(cb + code * 16);
        } else {
            constexpr int FPS = 8 / DIM;
            uint32_t o[4];
#pragma unroll
            for (int f = 0; f < FPS; f++) {
                const int bo = (s * FPS + f) * PB, wi = bo >> 5, bs = bo & 31;
                uint32_t v = bs + PB <= 32 ? c.w[j][wi] >> bs
                                           : __builtin_amdgcn_alignbit(c.w[j][wi + 1 < 4 * F::RL ? wi + 1 : wi],
                                                                       c.w[j][wi], (uint32_t)bs);
                v = __builtin_elementwise_min(v & ((1u << PB) - 1u), kcm1);
                if constexpr (DIM == 2) {
                    o[f] = *(const uint32_t*)(cb + v * 4);
                } else if constexpr (DIM == 4) {
                    const u32x2 t = *(const u32x2*)(cb + v * 8);
                    o[2 * f] = t.x;
                    o[2 * f + 1] = t.y;
                } else {
                    const u32x4 t = *(const u32x4*)(cb + v * 16);
                    o[0] = t.x; o[1] = t.y; o[2] = t.z; o[3] = t.w;
                }
            }
            return u32x4{o[0], o[1], o[2], o[3]};
        }
    };
    // x fragment of row block i, step s: row 32 i + l32, piece 4 h + s
    const uint32_t arow = (uint32_t)l32 * 128, asw = (uint32_t)(l32 >> 1) & 7u;
    uint32_t aoff[4];
#pragma unroll
    for (int s = 0; s < 4; s++) aoff[s] = arow + 16u * ((uint32_t)(4 * h + s) ^ asw);
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

    Codes cw = read_codes(0);
    settle(cw, 0);
    if constexpr (F::ahead(NB)) {
        // Stage t's MFMAs run beside stage t + 1's gathers (its codes landed a
        // stage earlier); the wait, the barrier and the next loads stand in
        // the middle of a stage, so the next stage's first x fragments are
        // read before this one ends.
        constexpr int Q = 4 * NB, D = 3;
        constexpr int MID = Q / 2 < Q - D ? Q / 2 : Q - D;     // before the next stage's first read
        u32x4 A[4];
        u32x4 B[2][2][4];                           // [stage parity][row block][step]
#pragma unroll
        for (int g = 0; g < 8; g++) B[0][g & 1][g >> 1] = gather(cw, g & 1, g >> 1);
#pragma unroll
        for (int q = 0; q < D; q++) {
            const int s = F::PACKED ? q % 4 : q / NB, i = F::PACKED ? q / 4 : q % NB;
            A[q % 4] = read_x(ar, i, s);
        }
        auto stage = [&](int t, auto par) {
            constexpr int c = decltype(par)::value;
            const unsigned char* base = ar + (t % S) * AB;
            const unsigned char* next = ar + ((t + 1) % S) * AB;
            const float sc0 = f16_to_f32((uint16_t)cw.sc[0]), sc1 = f16_to_f32((uint16_t)cw.sc[1]);
            cw = read_codes(t + 1);
            f32x16 P0, P1;
#pragma unroll
            for (int q = 0; q < Q; q++) {
                const int s = F::PACKED ? q % 4 : q / NB, i = F::PACKED ? q / 4 : q % NB;
                if (q == MID) {
                    vqg_wait<PER*(S - 3)>();        // this wave's x of stage t + 1 and codes of t + 2
                    lds_barrier();                  // and every wave's x; stage t - 1's buffer is free
                    issue_x(t + S - 1);
                    issue_c(t + S);
                }
                if (q == 0) settle(cw, t + 1);
#pragma unroll
                for (int g = 8 * q / Q; g < 8 * (q + 1) / Q; g++)
                    B[c ^ 1][g & 1][g >> 1] = gather(cw, g & 1, g >> 1);
                {
                    const int qn = (q + D) % Q;
                    const int sn = F::PACKED ? qn % 4 : qn / NB, in = F::PACKED ? qn / 4 : qn % NB;
                    A[(q + D) % 4] = read_x(q + D < Q ? base : next, in, sn);
                }
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (F::PACKED) {
                    const f32x16 zero = {};
                    P0 = vqg_mfma(A[q % 4], B[c][0][s], s ? P0 : zero);
                    P1 = vqg_mfma(A[q % 4], B[c][1][s], s ? P1 : zero);
                    if (s == 3) {
#pragma unroll
                        for (int r = 0; r < 16; r++) {
                            acc[i][0][r] = __builtin_fmaf(sc0, P0[r], acc[i][0][r]);
                            acc[i][1][r] = __builtin_fmaf(sc1, P1[r], acc[i][1][r]);
                        }
                    }
                } else {
                    acc[i][0] = vqg_mfma(A[q % 4], B[c][0][s], acc[i][0]);
                    acc[i][1] = vqg_mfma(A[q % 4], B[c][1][s], acc[i][1]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        int t = 0;
        for (; t + 1 < nk; t += 2) {
            stage(t, std::integral_constant<int, 0>());
            stage(t + 1, std::integral_constant<int, 1>());
        }
        if (t < nk) stage(t, std::integral_constant<int, 0>());
    } else if constexpr (!F::PACKED) {
        u32x4 B[2][2];                              // [step parity][row block]
        B[0][0] = gather(cw, 0, 0);
        B[0][1] = gather(cw, 1, 0);
        for (int t = 0; t < nk; t++) {
            vqg_wait<PER*(S - 2)>();                // this wave's x of stage t and codes of t + 1 are in LDS
            lds_barrier();                          // and every wave's x
            issue_x(t + S - 1);
            issue_c(t + S);
            const unsigned char* base = ar + (t % S) * AB;
            const Codes cn = read_codes(t + 1);
            // fragment q = s * NB + i of the stage, read D ahead of its MFMAs
            constexpr int Q = 4 * NB, D = Q < 4 ? Q - 1 : 3;
            u32x4 A[4];
#pragma unroll
            for (int q = 0; q < D; q++) A[q % 4] = read_x(base, q % NB, q / NB);
#pragma unroll
            for (int q = 0; q < Q; q++) {
                const int s = q / NB, i = q % NB, c = s & 1;
                if (i == 0) {                       // the next step's gathers
                    B[c ^ 1][0] = s < 3 ? gather(cw, 0, s + 1) : gather(cn, 0, 0);
                    B[c ^ 1][1] = s < 3 ? gather(cw, 1, s + 1) : gather(cn, 1, 0);
                }
                if (q + D < Q) A[(q + D) % 4] = read_x(base, (q + D) % NB, (q + D) / NB);
                __builtin_amdgcn_sched_barrier(0);
                acc[i][0] = vqg_mfma(A[q % 4], B[c][0], acc[i][0]);
                acc[i][1] = vqg_mfma(A[q % 4], B[c][1], acc[i][1]);
                __builtin_amdgcn_sched_barrier(0);
            }
            cw = cn;
        }
    } else {
        u32x4 B[2][4];
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int s = 0; s < 4; s++) B[j][s] = gather(cw, j, s);
        for (int t = 0; t < nk; t++) {
            vqg_wait<PER*(S - 2)>();
            lds_barrier();
            issue_x(t + S - 1);
            issue_c(t + S);
            const unsigned char* base = ar + (t % S) * AB;
            const float sc0 = f16_to_f32((uint16_t)cw.sc[0]), sc1 = f16_to_f32((uint16_t)cw.sc[1]);
            // fragment q = i * 4 + s, read D ahead of its MFMAs
            constexpr int Q = 4 * NB, D = 3;
            u32x4 A[4];
#pragma unroll
            for (int q = 0; q < D; q++) A[q % 4] = read_x(base, q / 4, q % 4);
#pragma unroll
            for (int i = 0; i < NB; i++) {
                f32x16 P0, P1;
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    const int q = 4 * i + s;
                    const f32x16 zero = {};
                    if (q + D < Q) A[(q + D) % 4] = read_x(base, (q + D) / 4, (q + D) % 4);
                    __builtin_amdgcn_sched_barrier(0);
                    P0 = vqg_mfma(A[q % 4], B[0][s], s ? P0 : zero);
                    P1 = vqg_mfma(A[q % 4], B[1][s], s ? P1 : zero);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (i == NB - 1) {                  // B's last use: the next stage's gathers go out
                    cw = read_codes(t + 1);
                    settle(cw, t + 1);
#pragma unroll
                    for (int j = 0; j < 2; j++)
#pragma unroll
                        for (int s = 0; s < 4; s++) B[j][s] = gather(cw, j, s);
                }
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    acc[i][0][r] = __builtin_fmaf(sc0, P0[r], acc[i][0][r]);
                    acc[i][1][r] = __builtin_fmaf(sc1, P1[r], acc[i][1][r]);
                }
            }
        }
    }

    // D of block (i, j): tile row 32 i + 8 (r / 4) + 4 h + r % 4, weight row of
    // block j.  Stored through a buffer view of y (a row past the tile or a
    // column past N at an offset past the view); one v_cvt_pk_bf16_f32 per two
    // values.
    float scl[2] = {1.f, 1.f};
    if constexpr (!F::PACKED) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int64_t n = col[j] < a.N ? col[j] : a.N - 1;
            scl[j] = f16_to_f32(a.sc[GLU ? j : 0][e0 + n]);
        }
    }
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
            if constexpr (GLU) {
                const bool ok = col[0] < a.N;
                // act = round(round(silu_f32(gate)) * up)
                const uint32_t g = cvt_pk_bf16(acc[i][0][r] * scl[0], acc[i][0][r + 1] * scl[0]);
                const uint32_t u = cvt_pk_bf16(acc[i][1][r] * scl[1], acc[i][1][r + 1] * scl[1]);
                uint32_t o = cvt_pk_bf16(silu_bf16r(lo16(g)) * lo16(u), silu_bf16r(hi16(g)) * hi16(u));
                if (a.y_f16) {
                    const vqg_f16x2 f = {(_Float16)lo16(o), (_Float16)hi16(o)};
                    o = __builtin_bit_cast(uint32_t, f);
                }
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const uint32_t off =
                        ok && rid[r + q] >= 0 ? (uint32_t)rid[r + q] * rowb + (uint32_t)col[0] * 2 : VQG_NONE;
                    __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(o >> (16 * q)), ry, (int)off, 0, 0);
                }
            } else {
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const uint32_t o = cvt_pk_bf16(acc[i][j][r] * scl[j], acc[i][j][r + 1] * scl[j]);
#pragma unroll
                    for (int q = 0; q < 2; q++) {
                        const uint32_t off = col[j] < a.N && rid[r + q] >= 0
                                                 ? (uint32_t)rid[r + q] * rowb + (uint32_t)col[j] * 2 : VQG_NONE;
                        __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(o >> (16 * q)), ry, (int)off, 0, 0);
                    }
                }
            }
        }
    }
    vqg_wait<0>();                                  // no load still writes LDS when the workgroup ends
}

template <int CB, int PB, int DIM, bool GLU>
__global__ __launch_bounds__(512, 1) void vq_gemm_kernel(VqgArgs a, int n_tiles, int tile_slots, int cbstride,
                                                         int two_cb) {
    using F = VqgFmt<CB, PB, DIM>;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ __align__(16) int32_t rid_s[VQG_RIDS];            // row id of tile row m (-1: none)
    // workgroup -> (tile, column block): the column blocks of a tile share an
    // XCD (workgroup i runs on XCD i % 8), where its x rows stay in L2
    const int id = (int)blockIdx.x, xcd = id & 7, kk = id >> 3;
    const int tile = 8 * (kk / n_tiles) + xcd;
    if (tile >= tile_slots) return;
    const int32_t* tp = a.tiles + 3 * (int64_t)tile;
    const int count = tp[2], start = tp[1];
    VqgTile tl = {tp[0], count, kk % n_tiles};
    if (count <= 0 || count > 32 * F::MAX_NB || tl.expert < 0 || tl.expert >= a.E) return;
    const int tid = threadIdx.x;
    if (tid < VQG_RIDS) rid_s[tid] = tid < count ? a.sorted[start + tid] : -1;
    lds_barrier();
    const int nb = (count + 31) / 32;
    if (nb == 1) vqg_body<F, CB, PB, DIM, GLU, 1>(a, tl, smem, rid_s, cbstride, two_cb);
    else if (nb == 2) vqg_body<F, CB, PB, DIM, GLU, 2>(a, tl, smem, rid_s, cbstride, two_cb);
    if constexpr (F::MAX_NB >= 3)
        if (nb == 3) vqg_body<F, CB, PB, DIM, GLU, 3>(a, tl, smem, rid_s, cbstride, two_cb);
    if constexpr (F::MAX_NB >= 4)
        if (nb == 4) vqg_body<F, CB, PB, DIM, GLU, 4>(a, tl, smem, rid_s, cbstride, two_cb);
    if constexpr (F::MAX_NB >= 5)
        if (nb == 5) vqg_body<F, CB, PB, DIM, GLU, 5>(a, tl, smem, rid_s, cbstride, two_cb);
}

__global__ __launch_bounds__(256) void vqg_to_f16_kernel(const u32x4* __restrict__ x, int64_t n8,
                                                         u32x4* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n8) return;
    const u32x4 v = x[i];
    u32x4 o;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const vqg_f16x2 p = {(_Float16)__uint_as_float(v[q] << 16), (_Float16)__uint_as_float(v[q] & 0xffff0000u)};
        o[q] = __builtin_bit_cast(uint32_t, p);
    }
    out[i] = o;
}

int vqg_cbstride(int kc, int dim) { return (kc * dim * 2 + 15) & ~15; }

// G: scale groups per row (packed; else 0)
size_t vqg_lds(int ring, int kc, int dim, bool two_cb, int G) {
    return (size_t)ring + (size_t)vqg_cbstride(kc, dim) * (two_cb ? 2 : 1) + VQG_WAVES * 2 * vqg_sc_bytes(G);
}

// the packed layouts compiled: f(PB, DIM)
#define KMI_VQG_PACKED(X)                                                                       \
    X(8, 2) X(9, 2) X(10, 2) X(11, 2) X(12, 2) X(8, 4) X(9, 4) X(10, 4) X(11, 4) X(12, 4)        \
    X(16, 4) X(8, 8) X(9, 8) X(10, 8) X(11, 8) X(12, 8) X(16, 8)

int vqg_ring(int code_bytes, int pack_bits, int dim) {
    if (code_bytes == 1) return VqgFmt<1, 8, 8>::max_ring();
    if (code_bytes == 2) return VqgFmt<2, 16, 8>::max_ring();
#define KMI_VQG_RING(PB_, D_) if (pack_bits == PB_ && dim == D_) return VqgFmt<0, PB_, D_>::max_ring();
    KMI_VQG_PACKED(KMI_VQG_RING)
#undef KMI_VQG_RING
    return 0;
}

template <int CB, int PB, int DIM>
int vqg_go(const VqgArgs& a, bool glu, int64_t tile_slots, hipStream_t st) {
    const bool two_cb = glu && a.cb[1] != a.cb[0];
    const size_t lds = vqg_lds(VqgFmt<CB, PB, DIM>::max_ring(), a.kc, DIM, two_cb, CB ? 0 : (int)(a.K / a.group));
    const int n_tiles = (int)ceil_div(a.N, glu ? 256 : 512);
    const int64_t wgs = 8 * n_tiles * ceil_div(tile_slots, 8);
    if (wgs >= (1LL << 31)) {
        set_error("vq_gemm: grid of %lld workgroups", (long long)wgs);
        return EINVAL_ARG;
    }
    const int cbs = vqg_cbstride(a.kc, DIM);
    if (glu) {
        allow_dynamic_lds_once((const void*)vq_gemm_kernel<CB, PB, DIM, true>);
        vq_gemm_kernel<CB, PB, DIM, true><<<(unsigned)wgs, 512, lds, st>>>(a, n_tiles, (int)tile_slots, cbs, two_cb);
    } else {
        allow_dynamic_lds_once((const void*)vq_gemm_kernel<CB, PB, DIM, false>);
        vq_gemm_kernel<CB, PB, DIM, false><<<(unsigned)wgs, 512, lds, st>>>(a, n_tiles, (int)tile_slots, cbs, two_cb);
    }
    return OK;
}

}  // namespace

bool vqg_supported(int code_bytes, int pack_bits, int dim, int group, int64_t E, int64_t N, int64_t K, int kc,
                   bool two_cb) {
    const int ring = vqg_ring(code_bytes, pack_bits, dim);
    if (!ring || K % VQG_BK || N <= 0) return false;
    if (code_bytes) {
        if (K % 128) return false;
    } else {
        // an expert's scales start on a word
        if (!(group == 64 || group == 128) || K % group || (N * (K / group)) % 2) return false;
    }
    return vqg_lds(ring, kc, dim, two_cb, code_bytes ? 0 : (int)(K / group)) + VQG_RIDS * 4 <= 160 * 1024;
}

int launch_vqg(const VqgArgs& a, int code_bytes, int pack_bits, int dim, bool glu, int64_t tile_slots,
               hipStream_t st) {
    const int64_t rb = code_bytes ? a.K / 8 * code_bytes : a.W * 4;
    if (!a.tiles || !a.sorted || a.lhs_div < 1 ||
        !vqg_supported(code_bytes, pack_bits, dim, a.group, a.E, a.N, a.K, a.kc, glu && a.cb[1] != a.cb[0])) {
        set_error("vq_gemm: shape outside the kernel");
        return EINVAL_ARG;
    }
    if (a.xrows * a.K * 2 >= (1LL << 31) || a.N * rb >= (1LL << 31) || a.rows * a.N * 2 >= (1LL << 31)) {
        set_error("vq_gemm: x, y or an expert's codes past 2 GiB");
        return EINVAL_ARG;
    }
    if (code_bytes == 1) return vqg_go<1, 8, 8>(a, glu, tile_slots, st);
    if (code_bytes == 2) return vqg_go<2, 16, 8>(a, glu, tile_slots, st);
#define KMI_VQG_GO(PB_, D_) if (pack_bits == PB_ && dim == D_) return vqg_go<0, PB_, D_>(a, glu, tile_slots, st);
    KMI_VQG_PACKED(KMI_VQG_GO)
#undef KMI_VQG_GO
    return EINVAL_ARG;
}

int launch_vqg_to_f16(const void* x, int64_t n, uint16_t* out, hipStream_t st) {
    vqg_to_f16_kernel<<<(unsigned)ceil_div(n / 8, 256), 256, 0, st>>>((const u32x4*)x, n / 8, (u32x4*)out);
    KMI_CHECK_LAUNCH("vqg_to_f16");
    return OK;
}

}  // namespace kmi
