// A prompt chunk's attention over the quantized KV cache (mlx-lm's
// quantized_scaled_dot_product_attention, .../_mlx_vlm/models/base.py:260-302)
// in one pass over the keys: scores, softmax and P V per tile of 64 keys, with
// no [rows, keys] score matrix in memory (the separate products write, mask,
// read and write it: at 512 queries x 32 heads over 8192 keys 268 MB each time).
//
// The query rows of a KV head (its rep query heads x L queries, consecutive in
// memory) are cut into tiles of 128: a workgroup of 4 waves, 32 rows each.
//   S^T = K Q^T: A is 32 keys of K, B the wave's 32 queries, both with the
//     head dimension as the contraction, so a lane holds 16 keys of one query
//     (keys 8 (r / 4) + 4 h + r % 4 of a block, h = lane / 32): softmax's
//     reductions run in registers, with one exchange between the two halves.
//     K's codes are exact in bf16: per group g the sum over the codes is
//     multiplied by the key's fp32 scale, and the group biases enter as one more
//     MFMA, sum_g b[key, g] * X[query, g] with X (the sum of the query over the
//     group) as three bf16 parts: scores are those of an fp32 dequantize.  They
//     are rounded to bf16 as the reference's are.
//   O^T = V^T P^T: a lane's 16 probabilities are B operands as they stand, with
//     V^T's keys stored in that order.  Each probability is multiplied by its
//     key's scale in fp32 and rounded once to bf16 (the reference rounds the
//     probability); V's codes, centred on 2^(bits - 1), are exact in bf16; the
//     biases' part of the sum is one fp32 dot product per query and group.
//     A row's running maximum moves only when a step passes it by 8 (a row
//     the step leaves alone is rescaled by 1).
// A tile's K codes and V^T codes are decoded to LDS once for all 128 rows
// (two buffers; the next tile's loads are in flight while a tile computes).
// Few rows leave CUs idle: the keys are then split, each split writing fp32
// sums with its maximum, merged by sdpa_merge.
// Measured, 512 queries x 32 heads over 4 KV heads, 8192 8-bit keys, D = 128: the
// separate products 515 us (233 scores, 152 softmax, 257 P V), one pass 131
// (vector instructions are issued 67% of the time, matrix
// cores busy 25%); 120 queries over 882 keys 118 -> 26 us (one launch's host
// work instead of three).  D = 256 holds one workgroup per CU: 512 queries x 16
// heads over 2 KV heads, 4096 keys 229 -> 129, 300 over 2000 117 -> 62.
// Chunks of 2048 queries over 4000 keys (few units, cut over all XCDs,
// dispatch.hpp; a unit per XCD in brackets): 32 heads over 4, D = 128 1006 -> 229 (435),
// 16 over 2, D = 256 765 -> 419 (1526).
#include "dispatch.hpp"
#include "qgemv_dl.hpp"
#include "../../include/knurlogic_amd.h"

namespace kmi {

namespace {

constexpr int SP_KT = 64;            // keys per tile
constexpr int SP_ROWS = 128;         // query rows per workgroup
constexpr float SP_LOG2E = 1.44269502f;

struct SpArgs {
    const uint16_t* q;               // [BHk, rows, D] bf16
    const uint32_t* w[2];            // K, V codes
    const uint16_t* s[2];
    const uint16_t* b[2];
    int64_t st[2][3][3];             // element strides (b, h, n) of w, s, b
    uint16_t* out;                   // [BHk, rows, D]
    float* po;                       // splits > 1: [splits, BHk, rows, D]
    float2* pm;                      // splits > 1: [splits, BHk, rows] (max, sum)
    int Hk, BHk, rows, L, N, causal;
    int splits, keys_per_split, row_tiles;
    float qscale;
};

__device__ __forceinline__ f32x16 sp_mfma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(a), as_bf16x8(b), c, 0, 0, 0);
}

__device__ __forceinline__ float sp_lo(uint32_t v) { return __uint_as_float(v << 16); }
__device__ __forceinline__ float sp_hi(uint32_t v) { return __uint_as_float(v & 0xffff0000u); }

// NW words of codes, natural order -> bf16 pairs
template <int BITS>
__device__ __forceinline__ u32x4 sp_codes8(uint32_t w0, uint32_t w1) {
    if constexpr (BITS == 4) return nib8_natural(w0);
    else return u32x4{bytes_to_bf16x2(w0, 0), bytes_to_bf16x2(w0, 2), bytes_to_bf16x2(w1, 0), bytes_to_bf16x2(w1, 2)};
}

// code j of 8 (in w0, w1), centred
template <int BITS>
__device__ __forceinline__ float sp_centred(uint32_t w0, uint32_t w1, int j) {
    if constexpr (BITS == 4) return (float)((w0 >> (4 * j)) & 15u) - 8.0f;
    else return (float)(int)(int8_t)(((j < 4 ? w0 : w1) ^ 0x80808080u) >> (8 * (j & 3)));
}

template <int BITS, int D>
struct SpShape {
    static constexpr int G = D / 64;                     // scale groups of 64
    static constexpr int KP = D * 2 + 16;                // bytes of a K row in LDS (padded)
    static constexpr int K_BYTES = SP_KT * KP;
    static constexpr int V_BYTES = D * SP_KT * 2;        // V^T rows of 64 keys
    static constexpr int KB_BYTES = SP_KT * (G > 2 ? 32 : 16);   // bias operand rows
    static constexpr int SC_BYTES = 3 * G * SP_KT * 4;   // K scales, V scales, V biases (centred), fp32
    static constexpr int STAGE = K_BYTES + V_BYTES + KB_BYTES + SC_BYTES;
    static constexpr int KW = D * BITS / 32 / 4;         // words of K codes per thread (a quarter row)
    static constexpr int NV = D / 128 > 0 ? D / 128 : 1; // (quad, octet) items per thread
    static constexpr int VW = BITS / 4;                  // words per 8 codes
    static constexpr int NS = (2 * G * SP_KT + 255) / 256;   // (scale, bias) pairs per thread
};

template <int BITS, int D>
__global__ __launch_bounds__(256, D > 128 ? 1 : 2) void sdpa_prefill_kernel(SpArgs a) {
    using S_ = SpShape<BITS, D>;
    constexpr int G = S_::G, KP = S_::KP, KW = S_::KW, NV = S_::NV, VW = S_::VW, NS = S_::NS, DB = D / 32;
    extern __shared__ __align__(16) unsigned char smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, h = lane >> 5;
    // workgroup -> (KV head and split, row tile): neighbours share an XCD,
    // whose L2 then holds their K and V
    const SpPlace wg = sp_place((int)blockIdx.x, a.BHk * a.splits, a.row_tiles);
    if (wg.unit < 0) return;
    const int unit = wg.unit, tile = wg.tile;
    const int head = unit / a.splits, split = unit % a.splits;
    const int64_t bi = head / a.Hk, hi = head % a.Hk;

    const int row = tile * SP_ROWS + wave * 32 + l32;
    const int rowc = row < a.rows ? row : a.rows - 1;
    // the last key this lane's query sees, and the last any of the tile's does
    const int vis = a.causal ? a.N - a.L + rowc % a.L : a.N - 1;
    const int r0 = tile * SP_ROWS, r1 = (r0 + SP_ROWS < a.rows ? r0 + SP_ROWS : a.rows) - 1;
    const int lmax = r1 / a.L > r0 / a.L ? a.L - 1 : r1 % a.L;
    const int tvis = a.causal ? a.N - a.L + lmax : a.N - 1;
    const int lmin = r1 / a.L > r0 / a.L ? 0 : r0 % a.L;
    const int tfull = a.causal ? a.N - a.L + lmin : a.N - 1;   // keys up to here are seen by every row
    const int kbeg = split * a.keys_per_split;
    int kend = kbeg + a.keys_per_split < a.N ? kbeg + a.keys_per_split : a.N;
    if (kend > tvis + 1) kend = tvis + 1;

    // ---- tile loads (registers), decode to LDS
    const unsigned char* kw = (const unsigned char*)(a.w[0] + bi * a.st[0][0][0] + hi * a.st[0][0][1]);
    const unsigned char* vw = (const unsigned char*)(a.w[1] + bi * a.st[1][0][0] + hi * a.st[1][0][1]);
    const int64_t kstride = a.st[0][0][2] * 4, vstride = a.st[1][0][2] * 4;
    const int kkey = tid >> 2, kpart = tid & 3;
    uint32_t rk[KW], rv[NV][4][VW];
    uint16_t rs[NS], rb[NS];
    const uint16_t* skp = a.s[0] + bi * a.st[0][1][0] + hi * a.st[0][1][1];
    const uint16_t* bkp = a.b[0] + bi * a.st[0][2][0] + hi * a.st[0][2][1];
    const uint16_t* svp = a.s[1] + bi * a.st[1][1][0] + hi * a.st[1][1][1];
    const uint16_t* bvp = a.b[1] + bi * a.st[1][2][0] + hi * a.st[1][2][1];
    auto load = [&](int k0) {
        {
            const int key = k0 + kkey < a.N ? k0 + kkey : a.N - 1;
            const unsigned char* p = kw + key * kstride + kpart * (KW * 4);
            if constexpr (KW == 2) {
                const u32x2 v = *(const u32x2*)p;
                rk[0] = v.x; rk[1] = v.y;
            } else {
#pragma unroll
                for (int i = 0; i < KW; i += 4) {
                    const u32x4 v = *(const u32x4*)(p + 4 * i);
                    rk[i] = v.x; rk[i + 1] = v.y; rk[i + 2] = v.z; rk[i + 3] = v.w;
                }
            }
        }
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const int item = tid + 256 * i, oct = item % (D / 8), quad = item / (D / 8);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int kq = k0 + 4 * (quad < 16 ? quad : 15) + j, key = kq < a.N ? kq : a.N - 1;
                const unsigned char* p = vw + key * vstride + oct * (VW * 4);
                if constexpr (VW == 2) {
                    const u32x2 v = *(const u32x2*)p;
                    rv[i][j][0] = v.x; rv[i][j][1] = v.y;
                } else rv[i][j][0] = *(const uint32_t*)p;
            }
        }
        // element e: (K, V)[e / (64 G)], key, group: its scale and bias
#pragma unroll
        for (int i = 0; i < NS; i++) {
            const int e = tid + 256 * i, t = e / (SP_KT * G), key = (e / G) % SP_KT, g = e % G;
            rs[i] = rb[i] = 0;
            if (e < 2 * SP_KT * G && k0 + key < a.N) {
                const int64_t n = k0 + key;
                const uint16_t* ps = (t ? svp : skp) + n * (t ? a.st[1][1][2] : a.st[0][1][2]) + g;
                const uint16_t* pb = (t ? bvp : bkp) + n * (t ? a.st[1][2][2] : a.st[0][2][2]) + g;
                rs[i] = *ps;
                rb[i] = *pb;
            }
        }
    };
    auto store = [&](int buf) {
        unsigned char* base = smem + buf * S_::STAGE;
        // K: this thread's quarter row
#pragma unroll
        for (int i = 0; i < KW / VW; i++)
            *(u32x4*)(base + kkey * KP + kpart * (D / 2) + 16 * i) = sp_codes8<BITS>(rk[VW * i], rk[VW * i + VW - 1]);
        // V^T: keys 4 quad .. + 3 of d = 8 oct + j at the operand's place: key
        // block u of 16 (quads 4 u .. + 3) gives lane half h quads 4 u + h and
        // 4 u + 2 + h, one 16-byte piece 2 u + h, swizzled over a row's 8 pieces
        unsigned char* vb = base + S_::K_BYTES;
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const int item = tid + 256 * i, oct = item % (D / 8), quad = item / (D / 8);
            if (D >= 128 || quad < 16) {
                const int piece = 2 * (quad >> 2) + (quad & 1), which = (quad >> 1) & 1;
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const int d = 8 * oct + j;
                    u32x2 v;
                    v.x = cvt_pk_bf16(sp_centred<BITS>(rv[i][0][0], rv[i][0][VW - 1], j),
                                      sp_centred<BITS>(rv[i][1][0], rv[i][1][VW - 1], j));
                    v.y = cvt_pk_bf16(sp_centred<BITS>(rv[i][2][0], rv[i][2][VW - 1], j),
                                      sp_centred<BITS>(rv[i][3][0], rv[i][3][VW - 1], j));
                    *(u32x2*)(vb + d * (SP_KT * 2) + ((piece ^ ((d + (d >> 3)) & 7)) * 16) + which * 8) = v;
                }
            }
        }
        // scales and biases
        unsigned char* kb = vb + S_::V_BYTES;
        float* sc = (float*)(kb + S_::KB_BYTES);
#pragma unroll
        for (int i = 0; i < NS; i++) {
            const int e = tid + 256 * i, t = e / (SP_KT * G), key = (e / G) % SP_KT, g = e % G;
            if (e >= 2 * SP_KT * G) continue;
            const float s = bf16_to_f32(rs[i]);
            if (t == 0) {
                // three slots of the bias operand: b times X's three parts (slots
                // 6 and 7 of a half are zero on the query's side)
                uint16_t* p = (uint16_t*)(kb + key * (G > 2 ? 32 : 16)) + (g >> 1) * 8 + (g & 1) * 3;
                p[0] = p[1] = p[2] = rb[i];
                sc[g * SP_KT + key] = s;
            } else {
                sc[(G + g) * SP_KT + key] = s;
                sc[(2 * G + g) * SP_KT + key] = __builtin_fmaf(BITS == 4 ? 8.f : 128.f, s, bf16_to_f32(rb[i]));
            }
        }
    };

    // ---- this lane's query: bf16(q * qscale) as B operands, X's parts
    u32x4 qf[D / 16], xf;
    {
        const uint16_t* qp = a.q + ((int64_t)head * a.rows + rowc) * D + 8 * h;
        float X[G];
#pragma unroll
        for (int g = 0; g < G; g++) X[g] = 0.f;
#pragma unroll
        for (int s = 0; s < D / 16; s++) {
            const u32x4 v = *(const u32x4*)(qp + 16 * s);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t w = cvt_pk_bf16(sp_lo(v[i]) * a.qscale, sp_hi(v[i]) * a.qscale);
                qf[s][i] = w;
                X[s / 4] += sp_lo(w) + sp_hi(w);
            }
        }
        uint16_t x3[4][3];
#pragma unroll
        for (int g = 0; g < 4; g++) {
            float v = g < G ? X[g < G ? g : 0] : 0.f;
            v += __shfl_xor(v, 32, 64);
#pragma unroll
            for (int t = 0; t < 3; t++) {
                x3[g][t] = f32_to_bf16(v);
                v -= bf16_to_f32(x3[g][t]);
            }
        }
        // half 0: groups 0, 1; half 1: groups 2, 3
        const int g0 = h * 2;
        auto pk = [](uint16_t lo, uint16_t hi16) { return (uint32_t)lo | ((uint32_t)hi16 << 16); };
        const uint32_t a0 = pk(x3[0][0], x3[0][1]), a1 = pk(x3[0][2], x3[1][0]), a2 = pk(x3[1][1], x3[1][2]);
        const uint32_t b0 = pk(x3[2][0], x3[2][1]), b1 = pk(x3[2][2], x3[3][0]), b2 = pk(x3[3][1], x3[3][2]);
        xf = u32x4{g0 ? b0 : a0, g0 ? b1 : a1, g0 ? b2 : a2, 0u};
    }

    f32x16 O[DB];
#pragma unroll
    for (int i = 0; i < DB; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) O[i][r] = 0.f;
    float bsum[G], lsum = 0.f, m = -__builtin_inff();      // m: -inf until the row sees a key
#pragma unroll
    for (int g = 0; g < G; g++) bsum[g] = 0.f;

    // the bias operand's unused slots must not hold NaN bits
    {
        for (int buf = 0; buf < 2; buf++) {
            uint32_t* p = (uint32_t*)(smem + buf * S_::STAGE + S_::K_BYTES + S_::V_BYTES);
            for (int i = tid; i < S_::KB_BYTES / 4; i += 256) p[i] = 0u;
        }
    }
    const int ntile = kend > kbeg ? (kend - kbeg + SP_KT - 1) / SP_KT : 0;
    if (ntile > 0) {
        load(kbeg);
        __syncthreads();
        store(0);
    }
    for (int t = 0; t < ntile; t++) {
        const int k0 = kbeg + t * SP_KT;
        __syncthreads();                             // tile t is in LDS, and tile t - 1's buffer is free
        const bool more = t + 1 < ntile;
        const unsigned char* base = smem + (t & 1) * S_::STAGE;
        const unsigned char* vb = base + S_::K_BYTES;
        const unsigned char* kbo = vb + S_::V_BYTES;
        const float* ksc = (const float*)(kbo + S_::KB_BYTES);
        const float* vsc = ksc + G * SP_KT;
        const float* vbi = vsc + G * SP_KT;

#pragma unroll 1
        for (int kb = 0; kb < 2; kb++) {
            // the next tile's loads go out half-way (fewer registers held)
            if (kb == 1 && more) load(k0 + SP_KT);
            __builtin_amdgcn_sched_barrier(0);
            // bias operand: key 32 kb + l32; with one or two groups half 1 holds none
            u32x4 bf = *(const u32x4*)(kbo + (32 * kb + l32) * (G > 2 ? 32 : 16) + (G > 2 ? 16 * h : 0));
            if (G <= 2 && h) bf = u32x4{0u, 0u, 0u, 0u};
            const f32x16 zero = {};
            f32x16 S = sp_mfma(bf, xf, zero);
#pragma unroll
            for (int g = 0; g < G; g++) {
                f32x16 P;
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    const u32x4 kf = *(const u32x4*)(base + (32 * kb + l32) * KP + (64 * g + 16 * s + 8 * h) * 2);
                    P = sp_mfma(kf, qf[4 * g + s], s ? P : zero);
                }
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const f32x4 sc = *(const f32x4*)(ksc + g * SP_KT + 32 * kb + 8 * q + 4 * h);
#pragma unroll
                    for (int j = 0; j < 4; j++) S[4 * q + j] = __builtin_fmaf(sc[j], P[4 * q + j], S[4 * q + j]);
                }
                __builtin_amdgcn_sched_barrier(0);   // one group's fragments in registers at a time
            }
            // round to bf16; hide keys past what the query sees
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const uint32_t w = cvt_pk_bf16(S[r], S[r + 1]);
                S[r] = sp_lo(w);
                S[r + 1] = sp_hi(w);
            }
            if (k0 + 32 * kb + 31 > tfull || k0 + 32 * kb + 32 > kend) {
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int key = k0 + 32 * kb + 8 * (r / 4) + 4 * h + r % 4;
                    if (key > vis || key >= kend) S[r] = -__builtin_inff();
                }
            }
            float mx = S[0];
#pragma unroll
            for (int r = 1; r < 16; r++) mx = __builtin_fmaxf(mx, S[r]);
            mx = __builtin_fmaxf(mx, __shfl_xor(mx, 32, 64));
            if (__any(mx > m + 8.0f)) {
                // per row: what a row's neighbours score does not move its maximum
                const float mn = mx > m + 8.0f ? mx : m;
                const float f = mn == m ? 1.0f : __builtin_amdgcn_exp2f((m - mn) * SP_LOG2E);
                m = mn;
                lsum *= f;
#pragma unroll
                for (int g = 0; g < G; g++) bsum[g] *= f;
#pragma unroll
                for (int i = 0; i < DB; i++)
#pragma unroll
                    for (int r = 0; r < 16; r++) O[i][r] *= f;
            }
            // e^(S - m): one multiply-add per score while the rounding of m log2(e)
            // is under 2^-16; rows that have seen no key and larger scores
            // subtract m first
            float mb = m * SP_LOG2E;
            if (__any(!(__builtin_fabsf(m) <= 256.0f))) {
                const float ms = m == -__builtin_inff() ? 0.0f : m;
#pragma unroll
                for (int r = 0; r < 16; r++) S[r] -= ms;
                mb = 0.0f;
            }
#pragma unroll
            for (int r = 0; r < 16; r++) {
                S[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(S[r], SP_LOG2E, -mb));
                lsum += S[r];
            }
#pragma unroll
            for (int g = 0; g < G; g++) {
                u32x4 pf[2];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int at = g * SP_KT + 32 * kb + 8 * q + 4 * h;
                    const f32x4 sc = *(const f32x4*)(vsc + at);
                    const f32x4 bb = *(const f32x4*)(vbi + at);
                    // P scaled (rounded once), and the biases' part: b centred, stored so
                    float v[4];
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        v[j] = S[4 * q + j] * sc[j];
                        bsum[g] = __builtin_fmaf(S[4 * q + j], bb[j], bsum[g]);
                    }
                    pf[q >> 1][2 * (q & 1)] = cvt_pk_bf16(v[0], v[1]);
                    pf[q >> 1][2 * (q & 1) + 1] = cvt_pk_bf16(v[2], v[3]);
                }
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int u = 0; u < 2; u++) {
                        const int db = 2 * g + i, d = 32 * db + l32, piece = 2 * (2 * kb + u) + h;
                        const u32x4 vf =
                            *(const u32x4*)(vb + d * (SP_KT * 2) + ((piece ^ ((d + (d >> 3)) & 7)) * 16));
                        O[db] = sp_mfma(vf, pf[u], O[db]);
                    }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (more) store((t + 1) & 1);
    }

    // ---- this lane's query: d = 32 db + 8 (r / 4) + 4 h + r % 4
    lsum += __shfl_xor(lsum, 32, 64);
#pragma unroll
    for (int g = 0; g < G; g++) bsum[g] += __shfl_xor(bsum[g], 32, 64);
    if (row >= a.rows) return;
    const int64_t at = (int64_t)head * a.rows + row;
    if (a.splits == 1) {
        const float inv = 1.0f / lsum;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float bs = bsum[db / 2];
                u32x2 v;
                v.x = cvt_pk_bf16((O[db][4 * q] + bs) * inv, (O[db][4 * q + 1] + bs) * inv);
                v.y = cvt_pk_bf16((O[db][4 * q + 2] + bs) * inv, (O[db][4 * q + 3] + bs) * inv);
                *(u32x2*)(a.out + at * D + 32 * db + 8 * q + 4 * h) = v;
            }
    } else {
        const int64_t ps = (int64_t)split * a.BHk * a.rows + at;
        if (h == 0) a.pm[ps] = float2{m, lsum};
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float bs = bsum[db / 2];
                *(f32x4*)(a.po + ps * D + 32 * db + 8 * q + 4 * h) =
                    f32x4{O[db][4 * q] + bs, O[db][4 * q + 1] + bs, O[db][4 * q + 2] + bs, O[db][4 * q + 3] + bs};
            }
    }
}

// out[row] = sum_s w_s o_s / sum_s w_s l_s, w_s = e^(m_s - m): a workgroup per
// row, its splits dealt to 256 / (D / 4) groups of threads (each sums its own in
// order, the groups' sums are added in order), so few rows' loads are in
// flight together: 128 rows of 50 splits, D = 256 25 us with a thread per 4
// columns, 5 here; but 16384 rows of 4 splits, D = 128 7 and 17 us.  (The whole
// calls of 800 rows per KV head x 900 keys, D = 64, 8 heads, 4 splits: 28 us by rows,
// 23 by columns; 256 rows x 1500 keys, D = 128, 1 head, 24 splits 14 and 19.)
constexpr int SP_MAX_SPLITS = 512;

template <int D>
__global__ __launch_bounds__(256) void sdpa_merge(const float* __restrict__ po, const float2* __restrict__ pm,
                                                  int splits, int64_t rows, uint16_t* __restrict__ out) {
    constexpr int CPR = D / 4, NG = 256 / CPR;
    __shared__ float wgt[SP_MAX_SPLITS];
    __shared__ f32x4 part[256];
    const int tid = threadIdx.x, lane = tid & 63, c = tid % CPR, g = tid / CPR;
    const int64_t row = blockIdx.x;
    // every wave forms m and sum_s w_s l_s
    float m = -__builtin_inff();
    for (int s = lane; s < splits; s += 64) m = __builtin_fmaxf(m, pm[s * rows + row].x);
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) m = __builtin_fmaxf(m, __shfl_xor(m, d, 64));
    float l = 0.f;
    for (int s = lane; s < splits; s += 64) {
        const float2 ml = pm[s * rows + row];
        const float f = __builtin_amdgcn_exp2f((ml.x - m) * SP_LOG2E);
        if (tid < 64) wgt[s] = f;
        l = __builtin_fmaf(f, ml.y, l);
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) l += __shfl_xor(l, d, 64);
    __syncthreads();
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int s = g; s < splits; s += NG) {
        const f32x4 v = *(const f32x4*)(po + (s * rows + row) * D + 4 * c);
        const float f = wgt[s];
#pragma unroll
        for (int j = 0; j < 4; j++) o[j] = __builtin_fmaf(f, v[j], o[j]);
    }
    part[tid] = o;
    __syncthreads();
    if (g > 0) return;
#pragma unroll
    for (int q = 1; q < NG; q++)
#pragma unroll
        for (int j = 0; j < 4; j++) o[j] += part[q * CPR + c][j];
    const float inv = 1.0f / l;
    u32x2 v;
    v.x = cvt_pk_bf16(o[0] * inv, o[1] * inv);
    v.y = cvt_pk_bf16(o[2] * inv, o[3] * inv);
    *(u32x2*)(out + row * D + 4 * c) = v;
}

// The same with a thread per 4 columns: many rows of few splits.
__global__ __launch_bounds__(256) void sdpa_merge_flat(const float* __restrict__ po, const float2* __restrict__ pm,
                                                  int splits, int64_t rows, int D, uint16_t* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int cpr = D / 4;
    if (i >= rows * cpr) return;
    const int64_t row = i / cpr;
    const int c = (int)(i % cpr);
    float m = -__builtin_inff();
    for (int s = 0; s < splits; s++) m = __builtin_fmaxf(m, pm[s * rows + row].x);
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    float l = 0.f;
    for (int s = 0; s < splits; s++) {
        const float2 ml = pm[s * rows + row];
        const float f = __builtin_amdgcn_exp2f((ml.x - m) * SP_LOG2E);
        const f32x4 v = *(const f32x4*)(po + (s * rows + row) * D + 4 * c);
        l = __builtin_fmaf(f, ml.y, l);
#pragma unroll
        for (int j = 0; j < 4; j++) o[j] = __builtin_fmaf(f, v[j], o[j]);
    }
    const float inv = 1.0f / l;
    u32x2 v;
    v.x = cvt_pk_bf16(o[0] * inv, o[1] * inv);
    v.y = cvt_pk_bf16(o[2] * inv, o[3] * inv);
    *(u32x2*)(out + row * D + 4 * c) = v;
}

struct SpPlan {
    int row_tiles, splits, keys_per_split;
    size_t ws;
};

// Key splits.  Until the grid has two workgroups per CU (D = 256: one), each
// split at least 256 keys; or, where that is a long chain on few CUs, the split
// with the least of: a workgroup's tiles of 64 keys (2.0 us each at D = 64, 2.8
// at 128, 6.5 at 256) in rounds of the CUs, and the merge (10 us of launch and
// host time, its bytes there and back at 3 TB/s), if it is 15% less by that
// count.  Device time of 256-key splits alone, with this, and of the separate
// products: 64 rows x 500 keys, 16 heads over 2, D = 256 59, 18, 24 us; 8 heads
// over 1, D = 128 26, 13, 21; 72 rows x 16000 keys, D = 256 68, 32, 46.
SpPlan sp_plan(int64_t BHk, int64_t rows, int64_t N, int64_t D) {
    SpPlan p;
    p.row_tiles = (int)ceil_div(rows, SP_ROWS);
    const int64_t wgs = BHk * p.row_tiles, slots = D > 128 ? 256 : 512, tiles = ceil_div(N, SP_KT);
    const double tile_us = D > 128 ? 6.5 : D > 64 ? 2.8 : 2.0, split_us = 0.05 + (double)(BHk * rows) * D * 8 / 3e6;
    auto cost = [&](int64_t per) {
        const int64_t s = ceil_div(tiles, per);
        return (double)ceil_div(wgs * s, slots) * per * tile_us + (s > 1 ? 10 + s * split_us : 0);
    };
    int64_t s0 = wgs < slots ? slots / wgs : 1;
    if (s0 > N / 256) s0 = N / 256 > 0 ? N / 256 : 1;
    int64_t best = ceil_div(ceil_div(N, s0), SP_KT);
    double best_us = cost(best) * 0.85;
    for (int64_t t = best;; t = t > 4 ? t * 3 / 4 : t - 1) {
        const int64_t s = ceil_div(tiles, t), even = ceil_div(tiles, s);
        if (s > SP_MAX_SPLITS) break;
        if (cost(even) < best_us) {
            best_us = cost(even);
            best = even;
        }
        if (t == 1) break;
    }
    p.keys_per_split = (int)(best * SP_KT);
    p.splits = (int)ceil_div(tiles, best);
    p.ws = p.splits > 1 ? (size_t)p.splits * BHk * rows * (D * 4 + 8) : 0;
    return p;
}

template <int BITS, int D>
int sp_go(const SpArgs& a, hipStream_t st) {
    const int64_t wgs = ((int64_t)a.BHk * a.splits + SP_XCDS) * a.row_tiles;
    if (wgs >= (1LL << 31)) {
        set_error("sdpa_prefill: grid of %lld workgroups", (long long)wgs);
        return EINVAL_ARG;
    }
    constexpr size_t lds = 2 * SpShape<BITS, D>::STAGE;
    allow_dynamic_lds_once((const void*)sdpa_prefill_kernel<BITS, D>);
    sdpa_prefill_kernel<BITS, D><<<SP_XCDS * sp_run(a.BHk * a.splits, a.row_tiles), 256, lds, st>>>(a);
    KMI_CHECK_LAUNCH("sdpa_prefill");
    return OK;
}

}  // namespace

}  // namespace kmi

using namespace kmi;

extern "C" {

size_t kmi_sdpa_prefill_workspace_bytes(int64_t B, int64_t H, int64_t Hk, int64_t L, int64_t N, int64_t D) {
    if (B <= 0 || H <= 0 || Hk <= 0 || H % Hk || L <= 0 || N <= 0 || D <= 0) return 0;
    return sp_plan(B * Hk, H / Hk * L, N, D).ws;
}

int kmi_sdpa_prefill(const void* q, int64_t B, int64_t H, int64_t L, int64_t D, const uint32_t* kw, const void* ks,
                     const void* kb, const uint32_t* vw, const void* vs, const void* vb, const int64_t* strides,
                     int64_t Hk, int64_t N, int group_size, int bits, float scale, int causal, void* out,
                     void* workspace, size_t workspace_bytes, void* stream) {
    clear_error();
    KMI_CHECK_ARG(B >= 1 && Hk >= 1 && H >= Hk && H % Hk == 0 && L >= 1 && N >= 1 && (D == 64 || D == 128 || D == 256),
                  "sdpa_prefill: bad sizes (head dim 64, 128 or 256)");
    KMI_CHECK_ARG(group_size == 64 && (bits == 4 || bits == 8), "sdpa_prefill: %d bits, group %d (4 or 8, 64)", bits,
                  group_size);
    KMI_CHECK_ARG(!causal || N >= L, "sdpa_prefill: causal over %lld keys with %lld queries", (long long)N,
                  (long long)L);
    KMI_CHECK_ARG(q && kw && ks && kb && vw && vs && vb && strides && out, "sdpa_prefill: null pointer");
    KMI_CHECK_ARG(N < (1LL << 30) && H / Hk * L < (1LL << 30) && B * Hk < (1LL << 24), "sdpa_prefill: too large");
    auto al16 = [](const void* p) { return ((uintptr_t)p & 15u) == 0; };
    bool ok = al16(q) && al16(out) && al16(kw) && al16(vw);
    SpArgs a = {};
    for (int t = 0; t < 2; t++)
        for (int c = 0; c < 3; c++)
            for (int i = 0; i < 3; i++) {
                a.st[t][c][i] = strides[(t * 3 + c) * 3 + i];
                if (c == 0 && a.st[t][c][i] % 4) ok = false;      // rows of codes at 16-byte addresses
            }
    KMI_CHECK_ARG(ok, "sdpa_prefill: q, out and rows of codes must be 16-byte aligned");
    const int64_t rows = H / Hk * L;
    const SpPlan p = sp_plan(B * Hk, rows, N, D);
    if (p.ws > 0 && (!workspace || workspace_bytes < p.ws || !al16(workspace))) {
        set_error("sdpa_prefill: workspace of %zu bytes needed, %zu given", p.ws, workspace_bytes);
        return EWORKSPACE;
    }
    a.q = (const uint16_t*)q; a.out = (uint16_t*)out;
    a.w[0] = kw; a.s[0] = (const uint16_t*)ks; a.b[0] = (const uint16_t*)kb;
    a.w[1] = vw; a.s[1] = (const uint16_t*)vs; a.b[1] = (const uint16_t*)vb;
    a.Hk = (int)Hk; a.BHk = (int)(B * Hk); a.rows = (int)rows; a.L = (int)L; a.N = (int)N; a.causal = causal ? 1 : 0;
    a.splits = p.splits; a.keys_per_split = p.keys_per_split; a.row_tiles = p.row_tiles;
    // mlx casts the Python scalar to the queries' dtype before `queries *= scale`
    uint32_t sb;
    __builtin_memcpy(&sb, &scale, 4);
    if ((sb & 0x7fffffffu) <= 0x7f800000u) sb = (sb + 0x7fffu + ((sb >> 16) & 1u)) & 0xffff0000u;
    __builtin_memcpy(&a.qscale, &sb, 4);
    a.po = (float*)workspace;
    a.pm = p.splits > 1 ? (float2*)((char*)workspace + (size_t)p.splits * a.BHk * rows * D * 4) : nullptr;
    hipStream_t st = (hipStream_t)stream;
    int rc = EINVAL_ARG;
    if (bits == 8) rc = D == 64 ? sp_go<8, 64>(a, st) : D == 128 ? sp_go<8, 128>(a, st) : sp_go<8, 256>(a, st);
    else rc = D == 64 ? sp_go<4, 64>(a, st) : D == 128 ? sp_go<4, 128>(a, st) : sp_go<4, 256>(a, st);
    if (rc) return rc;
    if (p.splits > 1) {
        const int64_t n = (int64_t)a.BHk * rows;
        if (p.splits <= 6 || n * (D / 4) >= (p.splits <= 12 ? 256 : 512) * 256)
            sdpa_merge_flat<<<(unsigned)ceil_div(n * (D / 4), 256), 256, 0, st>>>(a.po, a.pm, p.splits, n, (int)D, a.out);
        else if (D == 64) sdpa_merge<64><<<(unsigned)n, 256, 0, st>>>(a.po, a.pm, p.splits, n, a.out);
        else if (D == 128) sdpa_merge<128><<<(unsigned)n, 256, 0, st>>>(a.po, a.pm, p.splits, n, a.out);
        else sdpa_merge<256><<<(unsigned)n, 256, 0, st>>>(a.po, a.pm, p.splits, n, a.out);
        KMI_CHECK_LAUNCH("sdpa_merge");
    }
    return OK;
}

}  // extern "C"
