// qt_planes.h — f32 products on the bf16 matrix cores (gfx950), exact operands.
//
// An f32 value v is the sum of three bf16 planes exactly: v rounded to bf16, the rest rounded
// to bf16, and what then remains (at most 8 significant bits).  A product of two planes is
// exact in f32.  Of the nine plane products of an f32 product three lie below 2^-25 of it,
// under its own rounding; the other six are accumulated in f32, the smallest first.
#pragma once
#include "qt_attn_mf.h"

__device__ __forceinline__ uint32_t qt_bf16x2(float a, float b) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{a, b}), b2));
}
__device__ __forceinline__ float qt_bf_lo(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float qt_bf_hi(uint32_t u) { return __uint_as_float(u & 0xFFFF0000u); }

// the planes of 8 values; chk becomes NaN when a value has none (infinite, NaN, or past
// bf16's range after rounding) and stays as it is otherwise
__device__ __forceinline__ void qt_planes8(const float (&v)[8], qt_u32x4 (&p)[3], float &chk) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float a = v[2 * i], b = v[2 * i + 1];
        const uint32_t h = qt_bf16x2(a, b);
        const float ra = a - qt_bf_lo(h), rb = b - qt_bf_hi(h);
        const uint32_t m = qt_bf16x2(ra, rb);
        chk = fmaf(ra, 0.f, fmaf(rb, 0.f, chk));
        p[0][i] = h;
        p[1][i] = m;
        p[2][i] = qt_bf16x2(ra - qt_bf_lo(m), rb - qt_bf_hi(m));
    }
}

__device__ __forceinline__ void qt_planes8(const float (&v)[8], qt_u32x4 (&p)[3]) {
    float unused = 0.f;
    qt_planes8(v, p, unused);
}

// Activation planes in the matrix core's operand order, [k / 32][row tile][plane][64 lanes][8]
// with lane = row % 16 + 16 (k % 32 / 8): where (row, k) of plane 0 is; the planes are 512 apart.
__device__ __forceinline__ size_t qt_frag_at(int row_tiles, int row, int k) {
    return ((size_t)((k >> 5) * row_tiles + (row >> 4)) * 3) * 512 + ((row & 15) + 16 * ((k & 31) >> 3)) * 8 + (k & 7);
}

__device__ __forceinline__ qt_f32x4 qt_mma6(const qt_u32x4 (&a)[3], const qt_u32x4 (&b)[3], qt_f32x4 c) {
    c = qt_mfma_bf16(a[0], b[2], c);
    c = qt_mfma_bf16(a[2], b[0], c);
    c = qt_mfma_bf16(a[1], b[1], c);
    c = qt_mfma_bf16(a[0], b[1], c);
    c = qt_mfma_bf16(a[1], b[0], c);
    return qt_mfma_bf16(a[0], b[0], c);
}
