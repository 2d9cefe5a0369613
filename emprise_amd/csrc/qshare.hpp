// Loads of 64 consecutive columns of a quantised row, in either layout of layout.hpp.
#pragma once
#include "common.hpp"
#include "layout.hpp"

namespace emprise {
namespace {

typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
// rows of the unit-major layout start at any even address
typedef uint32_t u32x4u __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32u __attribute__((aligned(2)));

// Loads through global-address-space pointers (global_load_*, counted by vmcnt only).
#define QGLOBAL __attribute__((address_space(1)))
__device__ __forceinline__ uint4 gld16(const void* p) {
    const u32x4v v = *(const QGLOBAL u32x4v*)p;
    return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint4 gld16u(const void* p) {
    const u32x4u v = *(const QGLOBAL u32x4u*)p;
    return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint32_t gld4u(const void* p) { return *(const QGLOBAL u32u*)p; }
__device__ __forceinline__ uint32_t gld2(const void* p) { return *(const QGLOBAL uint16_t*)p; }
__device__ __forceinline__ uint32_t gld1(const void* p) { return *(const QGLOBAL uint8_t*)p; }

// A lane's share of one block of its row: columns 64q .. 64q+63.
template <int T> struct QRaw;
template <> struct QRaw<kQ6K> {
    uint32_t w[3][4];  // word p of unit 4q+j in w[p][j]
    uint32_t sc;       // the four units' int8 scales
    uint32_t d;        // fp16 block scale
};
template <> struct QRaw<kQ4K> {
    uint32_t w[2][4];  // the 32 nibbles of units 2q and 2q+1
    uint32_t sm[3];    // chunked: scale bytes, min nibbles; unit-major: three pairs of the 12 packed bytes
    uint32_t dd;       // fp16 d | fp16 dmin << 16
};

template <bool CH> __device__ __forceinline__ void q_load(QRaw<kQ6K>& r, const uint8_t* row, int nb, int b, int q) {
    if constexpr (CH) {
        const uint8_t* base = row + (size_t)(b >> 4) * 3360;
        const int l = 4 * (b & 15) + q;
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            const uint4 v = gld16(base + p * 1024 + 16 * l);
            r.w[p][0] = v.x, r.w[p][1] = v.y, r.w[p][2] = v.z, r.w[p][3] = v.w;
        }
        r.sc = gld4u(base + 3072 + 4 * l);
        r.d = gld2(base + 3328 + 2 * (b & 15));
    } else {
        const uint8_t* base = row + (size_t)b * 192 + 48 * q;
        uint32_t x[12];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            const uint4 v = gld16u(base + 16 * p);
            x[4 * p] = v.x, x[4 * p + 1] = v.y, x[4 * p + 2] = v.z, x[4 * p + 3] = v.w;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int p = 0; p < 3; ++p) r.w[p][j] = x[3 * j + p];
        r.sc = gld4u(row + (size_t)nb * 192 + 16 * b + 4 * q);
        r.d = gld2(row + (size_t)nb * 208 + 2 * b);
    }
}

template <bool CH> __device__ __forceinline__ void q_load(QRaw<kQ4K>& r, const uint8_t* row, int nb, int b, int q) {
    const uint8_t *c0, *c1, *s;
    if constexpr (CH) {
        const uint8_t* base = row + (size_t)(b >> 4) * 2304;
        c0 = base + 16 * (4 * (b & 15) + q);
        c1 = c0 + 1024;
        s = base + 2048 + 12 * (b & 15);
        r.sm[0] = gld2(s + 2 * q);
        r.sm[1] = gld1(s + 8 + q);
        r.sm[2] = 0;
        r.dd = gld4u(base + 2240 + 4 * (b & 15));
    } else {
        c0 = row + (size_t)b * 128 + 32 * q;
        c1 = c0 + 16;
        s = row + (size_t)nb * 128 + 12 * b;
        r.sm[0] = gld2(s + 2 * q);
        r.sm[1] = gld2(s + 2 * q + 4);
        r.sm[2] = gld2(s + 2 * max(q - 2, 0));
        r.dd = gld4u(row + (size_t)nb * 140 + 4 * b);
    }
    const uint4 v0 = gld16(c0), v1 = gld16(c1);
    r.w[0][0] = v0.x, r.w[0][1] = v0.y, r.w[0][2] = v0.z, r.w[0][3] = v0.w;
    r.w[1][0] = v1.x, r.w[1][1] = v1.y, r.w[1][2] = v1.z, r.w[1][3] = v1.w;
}

// The scale and min of units 2q (p = 0) and 2q+1 (p = 1) of a block (quant.cpp:48-52).
template <bool CH> __device__ __forceinline__ void q4_sm(const QRaw<kQ4K>& r, int q, int p, uint32_t& sc, uint32_t& mn) {
    if constexpr (CH) {
        const uint32_t b = (r.sm[0] >> (8 * p)) & 0xffu;
        sc = b & 63u;
        mn = ((b >> 6) << 4) | ((r.sm[1] >> (4 * p)) & 15u);
    } else {
        const uint32_t a = (r.sm[0] >> (8 * p)) & 0xffu, b = (r.sm[1] >> (8 * p)) & 0xffu, c = (r.sm[2] >> (8 * p)) & 0xffu;
        sc = q < 2 ? (a & 63u) : ((b & 15u) | ((c >> 6) << 4));
        mn = q < 2 ? (b & 63u) : ((b >> 4) | ((a >> 6) << 4));
    }
}

}  // namespace
}  // namespace emprise
