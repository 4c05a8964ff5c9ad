// gf16.h -- GF(2^16) products on packed words, shared by the packed-row and the
// K/V kernels: byte maps applied with v_perm_b32, and doublings for fields
// whose generator is 2.
#pragma once

#include "gf8.h"
#include "kvec_internal.h"

namespace kvec {

constexpr int kRs16Tab = 24;          // dwords per coefficient: 4 byte maps x 6

// Four words' low bytes into one register and their high bytes into another:
// b[0], b[1] for words 0-3 of the window, b[2], b[3] for words 4-7.
__device__ __forceinline__ void split_bytes(u32x4 x, uint32_t b[4]) {
    b[0] = __builtin_amdgcn_perm(x.y, x.x, 0x06040200u);
    b[1] = __builtin_amdgcn_perm(x.y, x.x, 0x07050301u);
    b[2] = __builtin_amdgcn_perm(x.w, x.z, 0x06040200u);
    b[3] = __builtin_amdgcn_perm(x.w, x.z, 0x07050301u);
}

__device__ __forceinline__ u32x4 join_bytes(const uint32_t a[4]) {
    return u32x4{__builtin_amdgcn_perm(a[1], a[0], 0x05010400u),
                 __builtin_amdgcn_perm(a[1], a[0], 0x07030602u),
                 __builtin_amdgcn_perm(a[3], a[2], 0x05010400u),
                 __builtin_amdgcn_perm(a[3], a[2], 0x07030602u)};
}

// acc ^ map_a(bytes of fa) ^ map_b(bytes of fb): six v_perm_b32, three 3-input XORs.
__device__ __forceinline__ uint32_t gf16_fma2(uint32_t acc, const Gf8Fields& fa, const uint32_t* ta,
                                              const Gf8Fields& fb, const uint32_t* tb) {
    const uint32_t p0 = __builtin_amdgcn_perm(ta[1], ta[0], fa.f0);
    const uint32_t p1 = __builtin_amdgcn_perm(ta[3], ta[2], fa.f1);
    const uint32_t p2 = __builtin_amdgcn_perm(ta[5], ta[4], fa.f2);
    const uint32_t p3 = __builtin_amdgcn_perm(tb[1], tb[0], fb.f0);
    const uint32_t p4 = __builtin_amdgcn_perm(tb[3], tb[2], fb.f1);
    const uint32_t p5 = __builtin_amdgcn_perm(tb[5], tb[4], fb.f2);
    return xor3(xor3(xor3(acc, p0, p1), p2, p3), p4, p5);
}

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef short i16x2 __attribute__((ext_vector_type(2)));

// Scalar doubling, for the check: x * 2 with reduction word `red`.
__host__ __device__ __forceinline__ uint16_t gf16_dbl(uint16_t x, uint16_t red) {
    return uint16_t((x << 1) ^ ((x & 0x8000u) ? red : 0u));
}

// Two packed words times 2; red2 holds the reduction word in both halves.
__device__ __forceinline__ uint32_t gf16_dbl2(uint32_t x, uint32_t red2) {
    const uint32_t sh = __builtin_bit_cast(uint32_t, u16x2(__builtin_bit_cast(u16x2, x) << 1));
    const uint32_t top = __builtin_bit_cast(uint32_t, i16x2(__builtin_bit_cast(i16x2, x) >> 15));
    return __builtin_amdgcn_bitop3_b32(sh, top, red2, 0x78);   // sh ^ (top & red2)
}

// (x * 2) ^ y
__device__ __forceinline__ uint32_t gf16_dbl2_xor(uint32_t x, uint32_t red2, uint32_t y) {
    const uint32_t sh = __builtin_bit_cast(uint32_t, u16x2(__builtin_bit_cast(u16x2, x) << 1));
    const uint32_t top = __builtin_bit_cast(uint32_t, i16x2(__builtin_bit_cast(i16x2, x) >> 15));
    return xor3(sh, top & red2, y);
}

// Times 4 in one step: a word v = t * 2^14 + low is v * 4 = (low << 2) ^ T[t]
// with T[t] = t * 2^16 reduced, t the two bits shifted out.  T fits the eight
// bytes one v_perm_b32 indexes: lo = T[0] | T[1] << 16, hi = T[2] | T[3] << 16,
// with T[1] = 2^16 reduced (the reduction word) and T[2] = 2^17 reduced (its
// double, reduced again when its top bit is set).
struct Gf16Quad {
    uint32_t lo, hi;
};
__host__ __device__ __forceinline__ Gf16Quad gf16_quad_table(uint16_t red) {
    const uint16_t r2 = gf16_dbl(red, red);
    return Gf16Quad{uint32_t(red) << 16, uint32_t(r2) | (uint32_t(uint16_t(red ^ r2)) << 16)};
}

// (x * 4) ^ y for two packed words: shift, the two top bits' byte selectors
// (2t, 2t + 1) by one packed multiply-add, the table lookup and a 3-input XOR
// (five VALU ops; two doublings and the XOR take seven).
__device__ __forceinline__ uint32_t gf16_quad2_xor(uint32_t x, Gf16Quad q, uint32_t y) {
    const u16x2 v = __builtin_bit_cast(u16x2, x);
    const uint32_t sh = __builtin_bit_cast(uint32_t, u16x2(v << 2));
    const u16x2 t = v >> 14;
    const uint32_t sel = __builtin_bit_cast(uint32_t, u16x2(t * u16x2{0x0202, 0x0202} + u16x2{0x0100, 0x0100}));
    return xor3(sh, __builtin_amdgcn_perm(q.hi, q.lo, sel), y);
}

// Four packed word pairs times alpha^e for alpha = 2 and 1 <= e <= 4 (e
// wave-uniform): one times-4 step when e >= 3, then one doubling (e odd) or
// one more times-4 step; straight-line code under two uniform branches.
__device__ __forceinline__ void gf16_step_pow(uint32_t (&a)[4], int e, uint32_t red2, Gf16Quad q) {
    if (e >= 3) {
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = gf16_quad2_xor(a[i], q, 0u);
    }
    if (e & 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = gf16_dbl2(a[i], red2);
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = gf16_quad2_xor(a[i], q, 0u);
    }
}

// a = a * alpha^e ^ y, as gf16_step_pow with the XOR in the last step.
__device__ __forceinline__ void gf16_step_pow_xor(uint32_t (&a)[4], int e, const uint32_t (&y)[4], uint32_t red2,
                                                  Gf16Quad q) {
    if (e >= 3) {
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = gf16_quad2_xor(a[i], q, 0u);
    }
    if (e & 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = gf16_dbl2_xor(a[i], red2, y[i]);
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = gf16_quad2_xor(a[i], q, y[i]);
    }
}

// Whether the pack and kvec_rs16_encode beat the one-pass encode, gs_rs16.hip.
bool rs16_ring_encode_faster(int k, int m, uint64_t Sb);

}  // namespace kvec
