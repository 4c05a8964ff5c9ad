// gs_star.h -- the star-diagonal P/Q code's word masks and star columns,
// shared by the packed-row and the K/V kernels.
#pragma once

#include "tile_engine.h"

namespace kvec {

// x % S with C semantics (the sign of x), dividing only when x is outside [0, S).
__device__ __forceinline__ int64_t cmod(int64_t x, int64_t S) {
    return (x >= 0 && x < S) ? x : x % S;
}

// v with its bytes 0..n-1 zeroed (n <= 0: v).
__device__ __forceinline__ u32x4 drop_low_bytes(u32x4 v, int n) {
    auto m = [&](int d) {
        const int k = n - 4 * d;   // bytes of dword d to clear
        return k <= 0 ? 0xFFFFFFFFu : (k >= 4 ? 0u : 0xFFFFFFFFu << (8 * k));
    };
    return u32x4{v.x & m(0), v.y & m(1), v.z & m(2), v.w & m(3)};
}

__device__ __forceinline__ u32x4 drop_word(u32x4 v, int64_t k) {
    if (k < 0 || k >= 8) return v;
    const uint32_t m = (k & 1) ? 0x0000FFFFu : 0xFFFF0000u;
    switch (k >> 1) {
        case 0: v.x &= m; break;
        case 1: v.y &= m; break;
        case 2: v.z &= m; break;
        default: v.w &= m; break;
    }
    return v;
}

// Per data row r < 16: the diagonal its star word lies on, (star_r + r) mod S
// with star_r = (star_base + r) % S, or -1 when the row skips nothing (C
// remainder: a negative star_base gives a negative star_r).  The same for
// every tile, so the host computes it once; the batched path runs only on
// row tensors below 2 GiB, so it fits 32 bits.
constexpr int kGsMaxRows = 16;   // rows of the one-tile kernels
struct GsStar {
    int32_t d[kGsMaxRows];
};

inline GsStar make_gs_star(int star_base, int64_t S) {
    GsStar star{};
    for (int r = 0; r < kGsMaxRows; ++r) {
        const int64_t sr = (int64_t(star_base) + r) % S;
        star.d[r] = sr < 0 ? -1 : int32_t((sr + r) % S);
    }
    return star;
}

// P and Q of 9 .. kGsMaxRows rows of S >= 64 words in a tensor whose bytes fit
// the kernels' resources, gs_kv.hip.
int gs_rdp_parity_wide(uint16_t* sh, int nd, int64_t S, int star_base, hipStream_t st, const char* what);
// The data row a recovery rebuilds, gs_xor_rdp.hip.
int gs_recover_row(int nd, int S, int star_base, int missing_a, int missing_b, const char* fn, int* row);

}  // namespace kvec
