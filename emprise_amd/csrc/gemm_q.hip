// Batched projections Y = X W^T with Q6_K / Q4_K weights on the fp16 matrix cores
// (Backend::linear_batch, reference backend.hpp:20-24 / the CUDA linear_q6_f32_batch,
// cuda.cpp:350-413), for every width and both weight layouts (layout.hpp).
//
// Both operands are exact in fp16 pieces, so the products are those of the FP32 path:
//
// - Weights. A Q6_K element is d * sc * (q - 32) with q a 6-bit code and sc an int8 unit
//   scale (quant.cpp:25-40); v = sc * (q - 32) is an integer of at most 13 bits, written
//   as v = vh + vl with vh = v rounded to fp16 and vl = v - vh (|vl| <= 1): both exact
//   fp16. A Q4_K element is (d * sc) * q - dmin * m (quant.cpp:41-61); v = sc * q is at
//   most 63 * 15 = 945, exact in fp16 as it stands. The block scales d (and dmin) of each
//   256 columns are applied in FP32 once per block.
// - Activations. Each 256-column block of a row of X is scaled by a power of two 2^-e
//   (exact) so that its largest magnitude lies in [2^14, 2^15) -- no fp16 overflow whatever
//   the activations; sums of 32 of them are carried 2^-6 times as large -- and split into xh =
//   fp16(x) and xl = fp16(x - xh), which carry 22 significant bits of every value down to 2^-16
//   of the block's largest. For up to 8 tokens, which FP32 matvecs served before, a third piece
//   carries the rest (split16).
//
// Per block the matrix cores accumulate, in FP32, sum v*xh + v*xl (+ vl*xh for Q6_K; the
// dropped vl*xl is below 2^-21 of the term) and 2^e * d times that is added to the row's
// FP32 accumulator; for Q4_K the min term -dmin * sum_u m_u * (sum of x over unit u) is
// one more product per block, with the unit sums split the same way.
//
// The weights never pass through LDS. The MFMA operand layout asks lane l for 8 columns of
// row l%16, and the order of the columns inside a block is free as long as both operands
// use the same one: lane (row, q = l/16) takes columns 64q .. 64q+63 of its row's block,
// which is what it gets from three (Q6_K) or two (Q4_K) 16-byte loads of codes, with its
// unit scales and the row's block scale beside them, and decodes them straight into
// operand registers in packed fp16 arithmetic, every step exact. Slice s of a block (one
// v_mfma_f32_16x16x32_f16 deep) is columns 64q + 8s .. +7 of each q. The activation pieces
// are stored by the split in that order, one 1 KiB operand after the other, so a step's
// share is a few contiguous runs and every LDS access is 16 bytes per lane in lane order.
//
// Three forms, by the number of tokens M (launch_type): up to 32 the weights' bytes bound
// the product and the waves stream them on their own (gemm_q16_few_kernel); up to 64, and
// where whole 256-row workgroups would leave CUs idle, gemm_q16_kernel; beyond that the
// matrix cores bound it (gemm_q16_wide_kernel). Where one workgroup per (rows, tokens) does
// not fill the chip the columns are cut into spans (gemm_q16_spans, a function of M and K
// alone, so that a row's sums do not depend on the rows it is stacked with), each span's
// sums a layer of scratch that gemm_q16_reduce_kernel adds up. Measured against a kernel
// that decoded the weights into LDS for 128 x 128 tiles (chunked layout) or dequantised
// them to FP32 (the others), graph replays over distinct weights, us, Q6_K gate+up rows
// 24576 x 4096 and down rows 4096 x 12288: 5 tokens 34 + 26 (58 + 34 as small-batch
// matvecs), 99 tokens 100 + 52 (the FFN 384 before, 158 now), 2048 tokens 950 + 503 (1276 +
// 620); Q4_K 12288 x 2048 and 2048 x 6144 at 700 tokens 148 + 85 (the FFN 1151 before, 219
// now).
//
// MFMA 16x16x32 f16 operand layout (lane l): A[i][k] with i = l % 16, k = 8*(l/16) + 0..7;
// B[k][j] with j = l % 16, the same k; D[i][j] in accumulator r with j = l % 16 and
// i = 4*(l/16) + r.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"
#include "layout.hpp"
#include "qshare.hpp"

namespace emprise {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
constexpr int kBlk = 256;             // columns per block
constexpr int kTileHalves = 16 * kBlk * 2;  // a 16-token tile's pieces of one block: 16 KiB

// ---- activations: fp16 hi/lo pieces of 2^-e * x, and (for Q4_K) of its 32-column sums ----

constexpr float kSumScale = 64.f;  // the unit sums are carried divided by this

// One token's 16 columns 16c .. 16c+15 of a block, by thread c of the token's 16 threads (a
// DPP row; all 16 call): slices 2(c%4), +1 of lane group q = c/4 into the tile's operands
// (slice s, piece p, lane l -> halves ((2s + p)*64 + l)*8 .. +7), 2^e, and with `sums` lane
// (i, q): the hi pieces of the sums over units 2q, 2q+1 (32 columns each), then their lo
// pieces.
//
// EIGHT: for at most 8 tokens, whose pieces fill the tile: token i's high pieces are row i of
// each slice's first operand, its low ones, carried 2^11 times as large, row i+8, and what
// they leave row i+8 of the second operand (its rows 0..7 are zero; the sums' pieces alike).
// So the products' rows 8..15 are the low part of tokens 0..7, to be added to rows 0..7, and
// x is carried whole, 24 bits of every value down to 2^-26 of the block's largest (of unit
// sums, 2^-20), as the FP32 matvecs that served these calls carried it. Error of an FFN's outputs
// at 5 tokens against 64 bits, Q4_K 512 -> 1536 -> 512 / 4096 -> 12288 -> 4096: 1.25e-7 / 1.37e-7
// (two pieces 1.65e-7 / 1.76e-7, the matvecs 1.30e-7 / 1.41e-7).
template <bool EIGHT>
__device__ __forceinline__ void split16(const float (&v)[16], int i, int c, _Float16* xf, float* xe, _Float16* xs,
                                        bool sums) {
    constexpr float kLow = 2048.f;
    const int q = c >> 2;
    float mx = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) mx = fmaxf(mx, fabsf(v[k]));
    mx = fmaxf(mx, dpp_f<0xb1, 0xf>(mx, mx));
    mx = fmaxf(mx, dpp_f<0x4e, 0xf>(mx, mx));
    mx = fmaxf(mx, dpp_f<0x141, 0xf>(mx, mx));
    mx = fmaxf(mx, dpp_f<0x140, 0xf>(mx, mx));
    int e = 0;
    if (mx > 0.f && mx < INFINITY) {
        (void)frexpf(mx, &e);      // mx = f * 2^e with f in [0.5, 1)
        e = max(e - 15, -126);     // mx * 2^-e in [2^14, 2^15)
    }
    const float up = ldexpf(1.f, -e);
    if (c == 0) {
        xe[i] = ldexpf(1.f, e);
        if constexpr (EIGHT) xe[i + 8] = ldexpf(1.f / kLow, e);
    }
    _Float16* dst = xf + (q * 16 + i) * 8;
    float s = 0.f;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        half8 hi, lo, rest;
        float w[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            w[k] = v[8 * h + k] * up;
            hi[k] = (_Float16)w[k];
            const float r = (w[k] - (float)hi[k]) * (EIGHT ? kLow : 1.f);
            lo[k] = (_Float16)r;
            rest[k] = (_Float16)(r - (float)lo[k]);
        }
        s += ((w[0] + w[1]) + (w[2] + w[3])) + ((w[4] + w[5]) + (w[6] + w[7]));
        _Float16* at = dst + (2 * (2 * (c & 3) + h)) * 512;
        *reinterpret_cast<half8*>(at) = hi;
        if constexpr (EIGHT) {
            *reinterpret_cast<half8*>(at + 64) = lo;
            *reinterpret_cast<half8*>(at + 512) = half8{};
            *reinterpret_cast<half8*>(at + 512 + 64) = rest;
        } else {
            *reinterpret_cast<half8*>(at + 512) = lo;
        }
    }
    if (sums) {
        s = (s + dpp_f<0xb1, 0xf>(0.f, s)) / kSumScale;  // the unit's two threads
        const float s1 = dpp_f<0x4e, 0xf>(0.f, s);    // lane group q's other unit
        if ((c & 3) == 0) {
            const _Float16 h0 = (_Float16)s, h1 = (_Float16)s1;
            half4* at = reinterpret_cast<half4*>(xs + (q * 16 + i) * 4);
            if constexpr (EIGHT) {
                const float r0 = (s - (float)h0) * kLow, r1 = (s1 - (float)h1) * kLow;
                const _Float16 l0 = (_Float16)r0, l1 = (_Float16)r1;
                at[0] = half4{h0, h1, (_Float16)0.f, (_Float16)0.f};
                at[8] = half4{l0, l1, (_Float16)(r0 - (float)l0), (_Float16)(r1 - (float)l1)};
            } else {
                at[0] = half4{h0, h1, (_Float16)(s - (float)h0), (_Float16)(s1 - (float)h1)};
            }
        }
    }
}

// 16 columns of token m (zero past M)
__device__ __forceinline__ void load16(float (&v)[16], const float* X, int m, int M, size_t ldx, int col) {
    if (m < M) {
        const floatx4* src = reinterpret_cast<const floatx4*>(X + (size_t)m * ldx + col);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const floatx4 f = src[k];
            v[4 * k] = f.x, v[4 * k + 1] = f.y, v[4 * k + 2] = f.z, v[4 * k + 3] = f.w;
        }
    } else {
#pragma unroll
        for (int k = 0; k < 16; ++k) v[k] = 0.f;
    }
}

// Workgroup = (16-token tile, block). xe[block][token]: 2^e; xs[block][tile][lane][4].
__global__ __launch_bounds__(256) void split_tiles_kernel(const float* __restrict__ X, int M, int ldx, int tiles,
                                                          _Float16* __restrict__ xf, float* __restrict__ xe,
                                                          _Float16* __restrict__ xs) {
    const int tile = blockIdx.x, blk = blockIdx.y, t = threadIdx.x, i = t >> 4, c = t & 15;
    float v[16];
    load16(v, X, tile * 16 + i, M, ldx, blk * kBlk + 16 * c);
    const size_t at = (size_t)blk * tiles + tile;
    split16<false>(v, i, c, xf + at * kTileHalves, xe + at * 16, xs + at * 256, xs != nullptr);
}

// ---- weights ---------------------------------------------------------------------------

// Two code bytes (bytes 0, 1 of w, or 2, 3 with hi) as the fp16 pair 1024 + q: each byte
// under an exponent byte 0x64 (v_perm_b32), which makes 1024 + q exact for q < 1024.
__device__ __forceinline__ half2v codes_1024(uint32_t w, bool hi) {
    return __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, w, hi ? 0x04030402u : 0x04010400u));
}
__device__ __forceinline__ half8 pack8(const uint32_t (&w)[4]) {
    return __builtin_bit_cast(half8, u32x4v{w[0], w[1], w[2], w[3]});
}

// The 16 columns of unit step j (64q + 16j .. +15) as two slices of operand registers.
// Q6_K: codes 0..3 in the low 6 bits of word 0, 4..7 of word 1, 8..11 of word 2, 12..15
// gathered from their top two bits; in packed fp16, each step exact: q - 32 = (1024 + q) -
// 1056; vh = fp16(v), v = sc * (q - 32); vl = fma(q - 32, sc, -vh), a small integer.
__device__ __forceinline__ void q6_unit(const QRaw<kQ6K>& r, int j, half8 (&hi)[2], half8 (&lo)[2]) {
    const uint32_t d0 = r.w[0][j], d1 = r.w[1][j], d2 = r.w[2][j];
    const uint32_t w[4] = {d0 & 0x3F3F3F3Fu, d1 & 0x3F3F3F3Fu, d2 & 0x3F3F3F3Fu,
                           ((d0 >> 6) & 0x03030303u) | ((d1 >> 4) & 0x0C0C0C0Cu) | ((d2 >> 2) & 0x30303030u)};
    const _Float16 s16 = (_Float16)(float)(int)(int8_t)(r.sc >> (8 * j));
    const half2v sc2 = {s16, s16}, off = {(_Float16)-1056.f, (_Float16)-1056.f};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        uint32_t ph[4], pl[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const half2v c = codes_1024(w[2 * h + (k >> 1)], k & 1) + off;
            const half2v vh = c * sc2;
            const half2v vl = __builtin_elementwise_fma(c, sc2, -vh);
            ph[k] = __builtin_bit_cast(uint32_t, vh);
            pl[k] = __builtin_bit_cast(uint32_t, vl);
        }
        hi[h] = pack8(ph);
        lo[h] = pack8(pl);
    }
}

// Q4_K: the low (j even) or high nibbles of unit 2q + j/2; v = (1024 + q) * sc - 1024 * sc
// in one fused step, exact: the product is below 1039 * 63 < 65504, the result at most 945.
template <bool CH> __device__ __forceinline__ void q4_unit(const QRaw<kQ4K>& r, int q, int j, half8 (&hi)[2]) {
    uint32_t sc, mn;
    q4_sm<CH>(r, q, j >> 1, sc, mn);
    const float scf = (float)sc;
    const _Float16 s16 = (_Float16)scf, b16 = (_Float16)(-1024.f * scf);
    const half2v sc2 = {s16, s16}, base = {b16, b16};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        uint32_t ph[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t nib = (r.w[j >> 1][2 * h + (k >> 1)] >> (4 * (j & 1))) & 0x0F0F0F0Fu;
            ph[k] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(codes_1024(nib, k & 1), sc2, base));
        }
        hi[h] = pack8(ph);
    }
}

// ---- the GEMM ------------------------------------------------------------------------

// Row r of the stacked weights.
template <int T> __device__ __forceinline__ const uint8_t* q_row(const QGemmArgs& a, int r, int nb) {
    const size_t row_bytes = (size_t)nb * (T == kQ6K ? 210 : 144);
    if (a.pair) return a.w[r & 1] + (size_t)(r >> 1) * row_bytes;
    int sg = 0;
    while (sg + 1 < a.nseg && r >= a.row0[sg + 1]) ++sg;
    return a.w[sg] + (size_t)(r - a.row0[sg]) * row_bytes;
}

// 16-byte piece v of block b's side data for mt token tiles from t0: 2^e, then the unit sums.
__device__ __forceinline__ uint4 q_side(const QGemmArgs& a, int tiles, int t0, int b, int v, int mt) {
    if (v < 4 * mt) return gld16(a.xe + ((size_t)b * tiles + min(t0 + (v >> 2), tiles - 1)) * 16 + 4 * (v & 3));
    const int u = v - 4 * mt;
    return gld16(a.xs + ((size_t)b * tiles + min(t0 + (u >> 5), tiles - 1)) * 256 + 8 * (u & 31));
}

// The block scales, and the Q4_K mins as a packed fp16 pair, kept past the raw words.
template <bool CH> __device__ __forceinline__ void q_block_scales(const QRaw<kQ6K>& r, int, uint32_t& d, uint32_t&) { d = r.d; }
template <bool CH> __device__ __forceinline__ void q_block_scales(const QRaw<kQ4K>& r, int q, uint32_t& d, uint32_t& mins) {
    uint32_t sc, m0, m1;
    q4_sm<CH>(r, q, 0, sc, m0);
    q4_sm<CH>(r, q, 1, sc, m1);
    d = r.dd;
    mins = __builtin_bit_cast(uint32_t, half2v{(_Float16)(-(float)m0), (_Float16)(-(float)m1)});
}

// Block end: acc += 2^e * (d * block products (- dmin * sum_u m_u * xsum_u)), products cleared.
// (2^e last: d * 2^e alone could overflow.)
template <int T, int RT, int MT>
__device__ __forceinline__ void q_block_end(const uint4* side, int lane, const uint32_t (&dblk)[RT],
                                            const uint32_t (&mins)[RT], floatx4 (&cb)[RT][MT], floatx4 (&acc)[RT][MT]) {
    const float4* E = reinterpret_cast<const float4*>(side);
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        if (MT * RT == 16 && m % 2 == 0) __builtin_amdgcn_sched_barrier(0);  // (registers: no further ahead)
        const float4 e4 = E[4 * m + (lane >> 4)];
        const float ev[4] = {e4.x, e4.y, e4.z, e4.w};
        half8 xsum = {};
        if constexpr (T == kQ4K) {
            const half4 p = reinterpret_cast<const half4*>(side + 4 * MT)[m * 64 + lane];
            xsum = half8{p[0], p[1], p[2], p[3], (_Float16)0.f, (_Float16)0.f, (_Float16)0.f, (_Float16)0.f};
        }
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            const float d = half_bits_to_float((uint16_t)(dblk[i] & 0xffffu));
            floatx4 cm = {0.f, 0.f, 0.f, 0.f};
            float dm = 0.f;
            if constexpr (T == kQ4K) {
                const half2v mm = __builtin_bit_cast(half2v, mins[i]);
                const half8 mv = {mm[0], mm[1], mm[0], mm[1], (_Float16)0.f, (_Float16)0.f, (_Float16)0.f, (_Float16)0.f};
                cm = __builtin_amdgcn_mfma_f32_16x16x32_f16(xsum, mv, cm, 0, 0, 0);
                dm = half_bits_to_float((uint16_t)(dblk[i] >> 16)) * kSumScale;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float t = d * cb[i][m][r];
                if constexpr (T == kQ4K) t = fmaf(dm, cm[r], t);
                acc[i][m][r] = fmaf(t, ev[r], acc[i][m][r]);
            }
            cb[i][m] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
}

// The products of slice h with token tiles m .. m+MP-1.
template <int T, int RT, int MP, int MT>
__device__ __forceinline__ void q_products(const half8 (&xh)[MP], const half8 (&xl)[MP], const half8 (&wh)[RT][2],
                                           const half8 (&wl)[RT][2], int h, int m, floatx4 (&cb)[RT][MT]) {
#pragma unroll
    for (int u = 0; u < MP; ++u)
#pragma unroll
        for (int i = 0; i < RT; ++i)
            cb[i][m + u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[u], wh[i][h], cb[i][m + u], 0, 0, 0);
    if constexpr (T == kQ6K) {
#pragma unroll
        for (int u = 0; u < MP; ++u)
#pragma unroll
            for (int i = 0; i < RT; ++i)
                cb[i][m + u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[u], wl[i][h], cb[i][m + u], 0, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < MP; ++u)
#pragma unroll
        for (int i = 0; i < RT; ++i)
            cb[i][m + u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[u], wh[i][h], cb[i][m + u], 0, 0, 0);
}

// A span's sums go to part[z][m][n]; with one layer, Y[m][n] directly. SwiGLU pairs: the
// gate (even n) and up (odd n) of one output sit in adjacent lanes; of accumulators r, r+1
// (rows m, m+1) the even lane writes row m and the odd lane row m+1, each receiving the one
// value it lacks through a lane swap, so every lane evaluates one silu(gate) * up
// (swiglu_kernel's form) per two entries.
template <int RT, int MT>
__device__ __forceinline__ void q_store(const QGemmArgs& a, int n0, int t0, int rj, int q, const floatx4 (&acc)[RT][MT]) {
    const bool odd = rj & 1;
    float* part = gridDim.z > 1 ? a.part + (size_t)blockIdx.z * a.M * a.N : nullptr;
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        const int n = n0 + 16 * i + rj;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int row_m = (t0 + m) * 16 + 4 * q;
#pragma unroll
            for (int r = 0; r < 4; r += 2) {
                const float v0 = acc[i][m][r], v1 = acc[i][m][r + 1];
                const int mr = row_m + r;
                if (part) {
                    if (n < a.N) {
                        if (mr < a.M) part[(size_t)mr * a.N + n] = v0;
                        if (mr + 1 < a.M) part[(size_t)(mr + 1) * a.N + n] = v1;
                    }
                } else if (a.pair) {
                    const float recv = dpp_f<0xb1, 0xf>(0.f, odd ? v0 : v1);  // quad_perm [1,0,3,2]
                    const float gate = odd ? recv : v0, up = odd ? v1 : recv;
                    const int mo = odd ? mr + 1 : mr;
                    if (mo < a.M && n < a.N) a.y[(size_t)mo * a.ldy + (n >> 1)] = siluf_(gate) * up;
                } else if (n < a.N) {
                    if (mr < a.M) a.y[(size_t)mr * a.ldy + n] = v0;
                    if (mr + 1 < a.M) a.y[(size_t)(mr + 1) * a.ldy + n] = v1;
                }
            }
        }
    }
}

// The general form. A workgroup of MT waves covers 16*MT weight rows x 16*MT tokens; all waves
// share the token operands, double-buffered in LDS one unit step (16 columns per lane) at a
// time, one barrier per step; a wave decodes each weight once for its 16*MT tokens.
// T: weight type; CH: chunked layout; MT: 16-token tiles; PF: the next block's weights are
// loaded a whole block ahead (a second register set) instead of during the block's last
// unit step. Grid: x = row groups, y = token groups, z = column spans. a.spans > 1 with one
// z layer runs the spans one after the other, adding them in the order the reduction
// would, so the results do not depend on which of the two forms ran. (The loops of one round
// are for the compiler's schedule. With / without them, us: FFN 4096 -> 12288 of 99 tokens,
// Q6_K 157.8 / 158.9, Q4_K 138.1 / 140.0; 2048 -> 6144 of 50, 50.2 / 50.4, 50.9 / 51.2; 1024 ->
// 3072 of 700, 233.9 / 234.5, 222.4 / 222.3.)
template <int T, bool CH, int MT, bool PF>
__global__ __launch_bounds__(MT * 64, 2) void gemm_q16_kernel(QGemmArgs a) {
    constexpr int TH = MT * 64;                         // threads
    constexpr int AV = MT * 4096 / 16;                  // 16-byte pieces of a step's operands
    constexpr int AN = AV / TH;
    constexpr int SV = MT * (T == kQ4K ? 36 : 4);       // of a block's side data: 2^e, then the unit sums
    constexpr int SN = (SV + TH - 1) / TH;
    constexpr int MP = 4;
    __shared__ __align__(16) uint4 As[2][AV];
    __shared__ __align__(16) uint4 Ss[2][SV];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 4, rj = lane & 15;
    const int tiles = (a.M + 15) >> 4, nb = a.K / kBlk;
    const int t0 = blockIdx.y * MT, n0 = (blockIdx.x * MT + wave) * 16;
    const int b0 = gridDim.z > 1 ? blockIdx.z * a.span : 0;
    const int b1 = gridDim.z > 1 ? min(b0 + a.span, nb) : nb;

    const uint8_t* row[1];  // (rows past N read the last row; their results are not stored)
#pragma unroll
    for (int i = 0; i < 1; ++i) row[0] = q_row<T>(a, min(n0 + 16 * i + rj, a.N - 1), nb);

    // step s (global numbering): unit step s % 4 of block s / 4
    uint4 ra[AN], rs[SN];
    auto load_a = [&](int s) {
        const int b = s / 4, j = s - b * 4;
#pragma unroll
        for (int k = 0; k < AN; ++k) {
            const int v = min(k * TH + tid, AV - 1), tile = v / 256, o = v - tile * 256;
            ra[k] = gld16(a.xf + ((size_t)b * tiles + min(t0 + tile, tiles - 1)) * kTileHalves + (size_t)(j * 256 + o) * 8);
        }
        if (j == 0) {
#pragma unroll
            for (int k = 0; k < SN; ++k) rs[k] = q_side(a, tiles, t0, b, min(k * TH + tid, SV - 1), MT);
        }
    };
    auto store_a = [&](int s, int buf) {
        const int b = s / 4, j = s - b * 4;
#pragma unroll
        for (int k = 0; k < AN; ++k) {
            const int v = k * TH + tid;
            As[buf][v] = ra[k];
        }
        if (j == 0) {
#pragma unroll
            for (int k = 0; k < SN; ++k) {
                const int v = k * TH + tid;
                if (v < SV) Ss[b & 1][v] = rs[k];
            }
        }
    };

    floatx4 cb[1][MT], acc[1][MT], tot[1][MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        cb[0][m] = acc[0][m] = floatx4{0.f, 0.f, 0.f, 0.f};
        tot[0][m] = floatx4{0.f, 0.f, 0.f, 0.f};
    }

    QRaw<T> raw[1], nxt[1];
    const int s0 = b0 * 4, s1 = b1 * 4;
    load_a(s0);
#pragma unroll
    for (int i = 0; i < 1; ++i) q_load<CH>(raw[0], row[0], nb, b0, q);
    store_a(s0, s0 & 1);
    load_a(min(s0 + 1, s1 - 1));
    lds_barrier();

    for (int b = b0; b < b1; ++b) {
        if constexpr (PF) {
#pragma unroll
            for (int i = 0; i < 1; ++i) q_load<CH>(nxt[0], row[0], nb, min(b + 1, b1 - 1), q);
        }
        uint32_t dblk[1], mins[1];
#pragma unroll
        for (int i = 0; i < 1; ++i) q_block_scales<CH>(raw[0], q, dblk[0], mins[0]);
#pragma unroll
        for (int js = 0; js < 4; ++js) {
            const int s = b * 4 + js, buf = s & 1;
            // the next step's operands go into the buffer that every wave finished with
            // before the last barrier; their loads had a whole step
            if (s + 1 < s1) store_a(s + 1, buf ^ 1);
            load_a(min(s + 2, s1 - 1));
            const half8* A = reinterpret_cast<const half8*>(As[buf]);
#pragma unroll
            for (int ju = 0; ju < 1; ++ju) {
                const int j = js + ju;
                half8 wh[1][2], wl[1][2];
#pragma unroll
                for (int i = 0; i < 1; ++i) {
                    if constexpr (T == kQ6K) q6_unit(raw[0], j, wh[0], wl[0]);
                    else q4_unit<CH>(raw[0], q, j, wh[0]);
                }
                if constexpr (!PF) {
                    if (j == 3) {
#pragma unroll
                        for (int i = 0; i < 1; ++i) q_load<CH>(raw[0], row[0], nb, min(b + 1, b1 - 1), q);
                    }
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    // MP token tiles at a time: consecutive MFMAs add to different accumulators
#pragma unroll
                    for (int m = 0; m < MT; m += MP) {
                        half8 xh[MP], xl[MP];
#pragma unroll
                        for (int u = 0; u < MP; ++u) {
                            xh[u] = A[(m + u) * 256 + (2 * h) * 64 + lane];
                            xl[u] = A[(m + u) * 256 + (2 * h + 1) * 64 + lane];
                        }
                        q_products<T, 1, MP, MT>(xh, xl, wh, wl, h, m, cb);
                    }
                }
            }
            if (js == 3) {
                q_block_end<T, 1, MT>(Ss[b & 1], lane, dblk, mins, cb, acc);
                if (gridDim.z == 1 && a.spans > 1 && ((b + 1) % a.span == 0 || b + 1 == b1)) {
#pragma unroll
                    for (int m = 0; m < MT; ++m)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            tot[0][m][r] += acc[0][m][r];
                            acc[0][m][r] = 0.f;
                        }
                }
            }
            lds_barrier();
        }
        if constexpr (PF) {
#pragma unroll
            for (int i = 0; i < 1; ++i) raw[0] = nxt[0];
        }
    }
    if (gridDim.z == 1 && a.spans > 1) {
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[0][m] = tot[0][m];
    }
    q_store<1, MT>(a, n0, t0, rj, q, acc);
}

// The forms for up to 32 tokens, where the weights' bytes are the bound: a workgroup splits
// its span of the activations itself (no pass before it), keeps all of it in LDS, and its
// waves then walk row tiles on their own.
constexpr int kFewSpan = 4;
constexpr int kEight = 8;  // tokens at most whose pieces share a 16-token tile (split16)
template <int T, int MT> struct Few {
    static constexpr int AV = MT * 1024;                        // 16-byte pieces of a block's operands
    static constexpr int SV = MT * (T == kQ4K ? 36 : 4);        // of its side data
    uint4 x[kFewSpan * AV], side[kFewSpan * SV];
};

// Blocks b0 .. b0+nbs-1 of the activations.
template <int T, int MT> __device__ __forceinline__ void few_stage(const QGemmArgs& a, int b0, int nbs, Few<T, MT>& lds) {
    using F = Few<T, MT>;
    if (MT == 1 && a.M <= kEight) {
        for (int t = threadIdx.x; t < nbs * 128; t += blockDim.x) {
            const int bl = t >> 7, i = (t >> 4) & 7, c = t & 15;
            float v[16];
            load16(v, a.x, i, a.M, a.ldx, (b0 + bl) * kBlk + 16 * c);
            uint4* side = lds.side + bl * F::SV;
            split16<true>(v, i, c, reinterpret_cast<_Float16*>(lds.x + bl * F::AV), reinterpret_cast<float*>(side),
                          reinterpret_cast<_Float16*>(side + 4), T == kQ4K);
        }
        return;
    }
    for (int t = threadIdx.x; t < nbs * MT * 256; t += blockDim.x) {
        const int u = t >> 8, i = (t >> 4) & 15, c = t & 15, bl = u / MT, m = u - bl * MT;
        float v[16];
        load16(v, a.x, m * 16 + i, a.M, a.ldx, (b0 + bl) * kBlk + 16 * c);
        uint4* side = lds.side + bl * F::SV;
        split16<false>(v, i, c, reinterpret_cast<_Float16*>(lds.x + bl * F::AV + m * 1024), reinterpret_cast<float*>(side + 4 * m),
                reinterpret_cast<_Float16*>(side + 4 * MT + 32 * m), T == kQ4K);
    }
}

// acc += the products of staged block bl.
//
// Three product sums per token tile, added at the block's end: the xh * vh of the even
// and of the odd slices, and the small terms -- shorter chains of FP32 additions
// (relative error against 64 bits at 5 tokens x 4096 columns, Q6_K / Q4_K: 1.03e-7 /
// 1.19e-7, with one sum and a float reduction 1.63e-7 / 1.92e-7, the FP32 matvec 1.83e-7
// / 1.19e-7)
template <int T, bool CH, int MT>
__device__ __forceinline__ void few_block(const QRaw<T>& raw, const Few<T, MT>& lds, int bl, int lane, floatx4 (&acc)[1][MT]) {
    using F = Few<T, MT>;
    const int q = lane >> 4;
    floatx4 cb[1][MT], c1[MT], cs[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) cb[0][m] = c1[m] = cs[m] = floatx4{0.f, 0.f, 0.f, 0.f};
    uint32_t dblk[1], mins[1];
    q_block_scales<CH>(raw, q, dblk[0], mins[0]);
    const half8* A = reinterpret_cast<const half8*>(lds.x + bl * F::AV);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        half8 wh[1][2], wl[1][2];
        if constexpr (T == kQ6K) q6_unit(raw, j, wh[0], wl[0]);
        else q4_unit<CH>(raw, q, j, wh[0]);
        half8 xh[2][MT], xl[2][MT];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                xh[h][m] = A[m * 1024 + (4 * j + 2 * h) * 64 + lane];
                xl[h][m] = A[m * 1024 + (4 * j + 2 * h + 1) * 64 + lane];
            }
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            cb[0][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[0][m], wh[0][0], cb[0][m], 0, 0, 0);
            c1[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[1][m], wh[0][1], c1[m], 0, 0, 0);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                cs[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[h][m], wh[0][h], cs[m], 0, 0, 0);
                if constexpr (T == kQ6K)
                    cs[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[h][m], wl[0][h], cs[m], 0, 0, 0);
            }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) cb[0][m][r] += c1[m][r] + cs[m][r];
    q_block_end<T, 1, MT>(lds.side + bl * F::SV, lane, dblk, mins, cb, acc);
}

// The tile's sums, of kEight tokens or fewer with their low part from the rows 8 further on
// (lanes 32 further on; what this leaves in those lanes is not stored).
template <int MT> __device__ __forceinline__ void few_finish(const QGemmArgs& a, floatx4 (&acc)[1][MT]) {
    if (MT > 1 || a.M > kEight) return;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[0][0][r]), __float_as_uint(acc[0][0][r]), false, false);
        acc[0][0][r] = __uint_as_float(s[0]) + __uint_as_float(s[1]);
    }
}

// No barrier after the staging, two blocks' weights in flight per wave; each tile's sums over
// the span go to part[z]. Grid: x = workgroups over the rows, z = spans of kFewSpan blocks.
template <int T, bool CH, int MT>
__global__ __launch_bounds__(1024) void gemm_q16_few_kernel(QGemmArgs a) {
    __shared__ __align__(16) Few<T, MT> lds;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 4, rj = lane & 15;
    const int nb = a.K / kBlk, b0 = blockIdx.z * kFewSpan, nbs = min(kFewSpan, nb - b0);
    const int waves = blockDim.x >> 6, ntiles = (a.N + 15) >> 4, stride = gridDim.x * waves;
    const int first = blockIdx.x * waves + wave;
    const int mine = first < ntiles ? (ntiles - first + stride - 1) / stride : 0;  // row tiles of this wave
    const int items = mine * nbs;

    struct At {
        int tile, b;           // row tile, block within the span
        const uint8_t* row;
    };
    auto seek = [&](At& p) { p.row = q_row<T>(a, min(p.tile * 16 + rj, a.N - 1), nb); };
    auto next = [&](At& p) {
        if (++p.b == nbs) {
            if (p.tile + stride < ntiles) {
                p.b = 0;
                p.tile += stride;
                seek(p);
            } else {
                p.b = nbs - 1;  // past the end: the last block again, never used
            }
        }
    };
    QRaw<T> r0, r1;
    At ld{min(first, ntiles - 1), 0, nullptr};
    seek(ld);
    q_load<CH>(r0, ld.row, nb, b0 + ld.b, q);
    next(ld);
    q_load<CH>(r1, ld.row, nb, b0 + ld.b, q);

    few_stage(a, b0, nbs, lds);
    __syncthreads();

    floatx4 acc[1][MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[0][m] = floatx4{0.f, 0.f, 0.f, 0.f};
    int tile = first, bl = 0;
    auto compute = [&](const QRaw<T>& raw) {
        few_block<T, CH, MT>(raw, lds, bl, lane, acc);
        if (++bl == nbs) {
            few_finish<MT>(a, acc);
            q_store<1, MT>(a, tile * 16, 0, rj, q, acc);
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[0][m] = floatx4{0.f, 0.f, 0.f, 0.f};
            bl = 0;
            tile += stride;
        }
    };
    for (int t = 0; t < items; t += 2) {
        compute(r0);
        next(ld);
        q_load<CH>(r0, ld.row, nb, b0 + ld.b, q);
        if (t + 1 < items) compute(r1);
        next(ld);
        q_load<CH>(r1, ld.row, nb, b0 + ld.b, q);
    }
}

// The same sums without scratch for them (a graph being captured, which cannot grow it): a
// workgroup stages one span after the other for its waves' row tiles and adds the spans'
// sums in registers, in gemm_q16_reduce_kernel's order and precision. Grid: x as above.
template <int T, bool CH, int MT>
__global__ __launch_bounds__(512) void gemm_q16_few_serial_kernel(QGemmArgs a) {
    __shared__ __align__(16) Few<T, MT> lds;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), q = lane >> 4, rj = lane & 15;
    const int nb = a.K / kBlk, waves = blockDim.x >> 6, ntiles = (a.N + 15) >> 4;
    for (int tile0 = blockIdx.x * waves; tile0 < ntiles; tile0 += gridDim.x * waves) {
        const int tile = tile0 + wave;  // (tiles past the last read the last row; their results are not stored)
        const uint8_t* row = q_row<T>(a, min(tile * 16 + rj, a.N - 1), nb);
        double tot[MT][4] = {};
        for (int b0 = 0; b0 < nb; b0 += kFewSpan) {
            const int nbs = min(kFewSpan, nb - b0);
            __syncthreads();
            few_stage(a, b0, nbs, lds);
            __syncthreads();
            floatx4 acc[1][MT];
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[0][m] = floatx4{0.f, 0.f, 0.f, 0.f};
            for (int bl = 0; bl < nbs; ++bl) {
                QRaw<T> raw;
                q_load<CH>(raw, row, nb, b0 + bl, q);
                few_block<T, CH, MT>(raw, lds, bl, lane, acc);
            }
            few_finish<MT>(a, acc);
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r) tot[m][r] += acc[0][m][r];
        }
        floatx4 acc[1][MT];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[0][m][r] = (float)tot[m][r];
        q_store<1, MT>(a, tile * 16, 0, rj, q, acc);
    }
}

// The form for more than 64 tokens: 8 waves of 32 rows x 128 tokens, one workgroup per CU.
// A step (one unit per lane, two slices) has a decode phase -- the operands of the next
// step to LDS, the weights of this one to registers, a finished block's scaling -- and a
// multiply phase of 96 (Q6_K) or 64 MFMAs with their LDS reads, a barrier after each.
// Waves 4..7 run one phase behind waves 0..3 (one of each on every SIMD), so that one
// group's vector work always runs beside the other's matrix work. Three operand buffers:
// both groups write step s+1 while the slower one still reads step s-1. Bound by the matrix
// cores and the registers: operands are read one pair ahead, not two, which for Q4_K spilled 33
// to 60 of them (2048 tokens x 12352 x 4096, Q4_K / Q6_K, 542 / 628 us, with two 813 / 639; the kernel of
// 128 x 128 tiles before this one 631 / 707). 2048 tokens x 24576 x 4096 in SwiGLU pairs 818 / 950 us:
// 1.0 / 1.3 PFLOP/s of fp16 products, where an 8192^3 fp16 product of the library holds 1.1.
template <int T, bool CH>
__global__ __launch_bounds__(512, 2) void gemm_q16_wide_kernel(QGemmArgs a) {
    constexpr int MT = 8, RT = 2, TH = 512, XD = 1;
    constexpr int AV = MT * 256, AN = AV / TH;
    constexpr int SV = MT * (T == kQ4K ? 36 : 4);
    __shared__ __align__(16) uint4 As[3][AV];
    __shared__ __align__(16) uint4 Ss[2][SV];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 4, rj = lane & 15;
    const int tiles = (a.M + 15) >> 4, nb = a.K / kBlk;
    const int t0 = blockIdx.y * MT, n0 = (blockIdx.x * 8 + wave) * (16 * RT);
    const int b0 = gridDim.z > 1 ? blockIdx.z * a.span : 0;
    const int b1 = gridDim.z > 1 ? min(b0 + a.span, nb) : nb;
    const uint8_t* row[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) row[i] = q_row<T>(a, min(n0 + 16 * i + rj, a.N - 1), nb);

    uint4 ra[AN], rs;
    uint32_t off[AN];  // of this thread's pieces of a step, in bytes
#pragma unroll
    for (int k = 0; k < AN; ++k) {
        const int v = k * TH + tid;
        off[k] = (uint32_t)min(t0 + (v >> 8), tiles - 1) * (kTileHalves * 2) + (v & 255) * 16;
    }
    auto load_a = [&](int s) {
        const int b = s >> 2, j = s & 3;
        const char* base = reinterpret_cast<const char*>(a.xf) + (size_t)b * tiles * (kTileHalves * 2) + j * 4096;
#pragma unroll
        for (int k = 0; k < AN; ++k) ra[k] = gld16(base + off[k]);
        if (j == 0 && tid < SV) rs = q_side(a, tiles, t0, b, tid, MT);
    };
    auto store_a = [&](int s, int buf) {
#pragma unroll
        for (int k = 0; k < AN; ++k) As[buf][k * TH + tid] = ra[k];
        if ((s & 3) == 0 && tid < SV) Ss[(s >> 2) & 1][tid] = rs;
    };

    floatx4 cb[RT][MT], acc[RT][MT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int m = 0; m < MT; ++m) cb[i][m] = acc[i][m] = floatx4{0.f, 0.f, 0.f, 0.f};

    QRaw<T> raw[RT];
    uint32_t dblk[RT], mins[RT];
    const int s0 = b0 * 4, s1 = b1 * 4;
    load_a(s0);
#pragma unroll
    for (int i = 0; i < RT; ++i) q_load<CH>(raw[i], row[i], nb, b0, q);
    store_a(s0, 0);
    load_a(s0 + 1);
    lds_barrier();
    if (wave >= 4) lds_barrier();
    int buf = 0;
    for (int b = b0; b < b1; ++b) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int s = b * 4 + j;
            const int nbuf = buf == 2 ? 0 : buf + 1;
            if (s + 1 < s1) store_a(s + 1, nbuf);
            load_a(min(s + 2, s1 - 1));
            if (j == 0) {
                if (b > b0) q_block_end<T, RT, MT>(Ss[(b - 1) & 1], lane, dblk, mins, cb, acc);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < RT; ++i) q_block_scales<CH>(raw[i], q, dblk[i], mins[i]);
            }
            half8 wh[RT][2], wl[RT][2];
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                if constexpr (T == kQ6K) q6_unit(raw[i], j, wh[i], wl[i]);
                else q4_unit<CH>(raw[i], q, j, wh[i]);
            }
            if (j == 3) {
#pragma unroll
                for (int i = 0; i < RT; ++i) q_load<CH>(raw[i], row[i], nb, min(b + 1, b1 - 1), q);
            }
            __builtin_amdgcn_sched_barrier(0);
            lds_barrier();
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(1);
            const half8* A = reinterpret_cast<const half8*>(As[buf]);
            // operand pairs (slice h, token tile m) in turn, each read XD pairs ahead of its
            // products: one wave of the SIMD multiplies, so nothing else hides its LDS reads
            half8 xh[XD + 1][1], xl[XD + 1][1];
            auto operands = [&](int k) {
                const int h = k / MT, m = k - h * MT;
                xh[k % (XD + 1)][0] = A[m * 256 + (2 * h) * 64 + lane];
                xl[k % (XD + 1)][0] = A[m * 256 + (2 * h + 1) * 64 + lane];
            };
#pragma unroll
            for (int k = 0; k < XD; ++k) operands(k);
#pragma unroll
            for (int k = 0; k < 2 * MT; ++k) {
                if (k + XD < 2 * MT) operands(k + XD);
                __builtin_amdgcn_sched_barrier(0);
                q_products<T, RT, 1, MT>(xh[k % (XD + 1)], xl[k % (XD + 1)], wh, wl, k / MT, k % MT, cb);
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
            lds_barrier();
            __builtin_amdgcn_sched_barrier(0);
            buf = nbuf;
        }
    }
    if (wave < 4) lds_barrier();
    q_block_end<T, RT, MT>(Ss[(b1 - 1) & 1], lane, dblk, mins, cb, acc);
    q_store<RT, MT>(a, n0, t0, rj, q, acc);
}

// Y[m][n] = sum over the spans, in order, in S (double for the form for few tokens, whose
// spans are short; float where the spans may also have been added in registers); SwiGLU
// pairs as above.
template <class S> __global__ __launch_bounds__(256) void gemm_q16_reduce_kernel(QGemmArgs a) {
    const int m = blockIdx.y, cols = a.pair ? a.N / 2 : a.N;
    const int n = blockIdx.x * 256 + threadIdx.x;
    if (n >= cols) return;
    const size_t layer = (size_t)a.M * a.N;
    if (a.pair) {
        const float2* p = reinterpret_cast<const float2*>(a.part + (size_t)m * a.N + 2 * n);
        S g = 0, u = 0;
        for (int z = 0; z < a.spans; ++z) {
            const float2 v = p[z * (layer / 2)];
            g += v.x;
            u += v.y;
        }
        a.y[(size_t)m * a.ldy + n] = siluf_((float)g) * (float)u;
    } else {
        const float* p = a.part + (size_t)m * a.N + n;
        S v = 0;
        for (int z = 0; z < a.spans; ++z) v += p[z * layer];
        a.y[(size_t)m * a.ldy + n] = (float)v;
    }
}

hipError_t launch_reduce(const QGemmArgs& a, int layers, hipStream_t stream) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || layers == 1) return e;
    const dim3 grid(((a.pair ? a.N / 2 : a.N) + 255) / 256, a.M);
    if (gemm_q16_few(a.M)) launch_kernel(gemm_q16_reduce_kernel<double>, grid, dim3(256), 0, stream, a);
    else launch_kernel(gemm_q16_reduce_kernel<float>, grid, dim3(256), 0, stream, a);
    return hipGetLastError();
}

constexpr int kCUs = 256;

// Token tiles per workgroup for M tokens.
int tiles_for(int M) { return M <= 16 ? 1 : M <= 32 ? 2 : M <= 64 ? 4 : 8; }

// One workgroup per CU over all the spans; the waves of each share its row tiles evenly (24576
// rows of 4096 and 16 tokens: 12 waves with two tiles each 37.9 us with the reduction, two
// 8-wave workgroups on half of the CUs 42.7).
template <int T, bool CH, int MT> hipError_t launch_few(const QGemmArgs& a, int layers, hipStream_t stream) {
    const int ntiles = (a.N + 15) / 16, gx = std::min(std::max(1, kCUs / layers), ntiles);
    const int most = layers == a.spans ? 16 : 8;  // waves per workgroup
    const int per = (ntiles + gx - 1) / gx, rounds = (per + most - 1) / most, waves = (per + rounds - 1) / rounds;
    const dim3 grid((ntiles + waves * rounds - 1) / (waves * rounds), 1, layers), block(waves * 64);
    if (layers == a.spans) launch_kernel(gemm_q16_few_kernel<T, CH, MT>, grid, block, 0, stream, a);
    else launch_kernel(gemm_q16_few_serial_kernel<T, CH, MT>, grid, block, 0, stream, a);
    return launch_reduce(a, layers, stream);
}

// Workgroups of mt token tiles x `rows` weight rows.
template <class F>
hipError_t launch_grid(F kernel, int mt, int rows, int threads, const QGemmArgs& a, int layers, hipStream_t stream) {
    const dim3 grid((a.N + rows - 1) / rows, ((a.M + 15) / 16 + mt - 1) / mt, layers);
    if (grid.y > 65535) return hipErrorInvalidValue;
    launch_kernel(kernel, grid, dim3(threads), 0, stream, a);
    return launch_reduce(a, layers, stream);
}

template <int T, bool CH, int MT, bool PF> hipError_t launch_form(const QGemmArgs& a, int layers, hipStream_t stream) {
    return launch_grid(gemm_q16_kernel<T, CH, MT, PF>, MT, MT * 16, MT * 64, a, layers, stream);
}

template <int T, bool CH> hipError_t launch_type(const QGemmArgs& a, int layers, hipStream_t stream) {
    const int mt = tiles_for(a.M);
    if (mt == 1) return launch_few<T, CH, 1>(a, layers, stream);
    if (mt == 2) return launch_few<T, CH, 2>(a, layers, stream);
    if (mt == 4) return launch_form<T, CH, 4, true>(a, layers, stream);
    // 256 rows per workgroup, or 128 where that fills the last round of workgroups better
    // (a workgroup of half the rows takes a bit over half the time)
    const int groups = ((a.M + 127) / 128) * layers;
    const int wide = (groups * ((a.N + 255) / 256) + kCUs - 1) / kCUs;
    const int half = (groups * ((a.N + 127) / 128) + kCUs - 1) / kCUs;
    if (half * 6 < wide * 10 || (layers == 1 && a.spans > 1) || a.M > (1 << 22))
        return launch_form<T, CH, 8, false>(a, layers, stream);
    return launch_grid(gemm_q16_wide_kernel<T, CH>, 8, 256, 512, a, layers, stream);
}

}  // namespace

size_t gemm_q16_split_bytes(int M, int K, bool sums) {
    const size_t tiles = (size_t)(M + 15) / 16, nb = K / kBlk;
    return tiles * nb * (kTileHalves * sizeof(_Float16) + 16 * sizeof(float) + (sums ? 512 : 0));
}

hipError_t launch_gemm_q16_split(const float* X, int M, int K, int ldx, void* scratch, bool sums, QGemmArgs* a,
                                 hipStream_t stream) {
    if (M < 1 || K < kBlk || K % kBlk || ldx < K || ldx % 4 || reinterpret_cast<uintptr_t>(X) % 16)
        return hipErrorInvalidValue;
    const int tiles = (M + 15) / 16, nb = K / kBlk;
    if (nb > 65535) return hipErrorInvalidValue;
    _Float16* xf = static_cast<_Float16*>(scratch);
    float* xe = reinterpret_cast<float*>(xf + (size_t)tiles * nb * kTileHalves);
    _Float16* xs = sums ? reinterpret_cast<_Float16*>(xe + (size_t)tiles * nb * 16) : nullptr;
    launch_kernel(split_tiles_kernel, dim3(tiles, nb), dim3(256), 0, stream, X, M, ldx, tiles, xf, xe, xs);
    a->xf = reinterpret_cast<const uint16_t*>(xf);
    a->xe = xe;
    a->xs = reinterpret_cast<const uint16_t*>(xs);
    a->M = M;
    a->K = K;
    return hipGetLastError();
}

bool gemm_q16_few(int M) { return M <= 32; }

// Column spans of a product with M tokens and K columns. The rows may not enter (a row's sums
// are the same bits whichever rows share its launch), so they are guessed from K. Wide inputs
// are taken for those of down projections, with K/3 rows, and get spans for one workgroup of 128
// x 128 per CU; narrower ones for the hidden state, whose projections have more rows and pay for
// each span with partial sums. Where widths may be either, few spans are the smaller loss: FFNs
// at 6144 hidden values or more are rare, and below that both kinds occur. us with few spans / with
// the wide rule's, at 300 and 700 tokens: FFN 4096 -> 5632 -> 4096, Q4_K, 700 only, 378 / 447; 4096 ->
// 5120 167 / 190 at 300; 5120 columns x 30720 rows, Q6_K, 350 / 437 and 606 / 759; but FFN 2048 -> 5888
// 174 / 138 and 260 / 216, 1536 -> 4608 120 / 96 and 175 / 130 (rows near K/3, which the line gives up).
int gemm_q16_spans(int M, int K) {
    const int nb = K / kBlk, groups = (M + 127) / 128;
    int spans;
    if (M <= 64) spans = (nb + kFewSpan - 1) / kFewSpan;
    else if (K >= 6144) spans = std::max(1, 3 * 128 * kCUs / K / groups);
    else spans = groups == 1 ? 4 : groups <= 4 ? 2 : 1;
    spans = std::max(1, std::min(spans, nb / 2));
    const int span = (nb + spans - 1) / spans;  // blocks in each but the last
    return (nb + span - 1) / span;
}

int gemm_q16_layers(int M, int N, int K) {
    const int spans = gemm_q16_spans(M, K), mt = tiles_for(M);
    if (spans == 1) return 1;
    // the spans can also run in one workgroup after the other: with enough rows for a full
    // chip, or very many partial sums, those need not go through memory
    if (mt >= 4 && (N >= 65536 || (size_t)spans * M * N > (size_t(64) << 20))) return 1;
    return spans;
}

hipError_t launch_gemm_q16(uint32_t type, QGemmArgs a, hipStream_t stream) {
    if ((type != kQ6K && type != kQ4K) || a.M < 1 || a.N < 1 || a.K % kBlk || a.nseg < 1 || a.nseg > kMaxSeg ||
        a.row0[0] != 0 || a.row0[a.nseg] != a.N || (!gemm_q16_few(a.M) && (!a.xf || (type == kQ4K && !a.xs))))
        return hipErrorInvalidValue;
    if (a.pair ? (a.nseg != 2 || a.N % 2 || a.row0[1] * 2 != a.N || a.ldy < a.N / 2) : a.ldy < a.N)
        return hipErrorInvalidValue;
    const int nb = a.K / kBlk, layers = a.part ? gemm_q16_layers(a.M, a.N, a.K) : 1;
    a.spans = gemm_q16_spans(a.M, a.K);
    a.span = (nb + a.spans - 1) / a.spans;
    if (gemm_q16_few(a.M) && a.span > kFewSpan) return hipErrorInvalidValue;
    if (layers > 1 && a.M > 65535) return hipErrorInvalidValue;
    const bool ch = chunked_cols(a.K);
    if (type == kQ6K) return ch ? launch_type<kQ6K, true>(a, layers, stream) : launch_type<kQ6K, false>(a, layers, stream);
    return ch ? launch_type<kQ4K, true>(a, layers, stream) : launch_type<kQ4K, false>(a, layers, stream);
}

}  // namespace emprise
