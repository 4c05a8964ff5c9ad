// kv_stream.h -- the coding stream read from, or written to, K and V where
// they lie.
//
// The reference's wrappers lay K and V out as one stream before they code it
// (torch permutes and copies, then a pack).  The kernels here address the
// stream's bytes in K and V themselves: stream bytes [0, kb) are K's and
// [kb, 2 kb) are V's, either in memory order (FLAT: contiguous K and V) or
// token major, [T][B][H][D] of tensors indexed [B][H][T][D] with any strides
// over B, H and T.  A head's D values are contiguous, a multiple of 16 bytes
// long and 16-byte aligned, so every aligned 16-byte chunk of the stream is
// one aligned chunk of K, one of V, or past both.
#pragma once

#include "tile_engine.h"

namespace kvec {

struct KvStream {
    uint8_t* K;
    uint8_t* V;
    uint32_t kb;           // bytes of K, and of V; < 2^30
    uint32_t ext;          // bytes from K's (V's) first byte to its last, < 2^31
    uint32_t sB, sH, sT;   // byte strides (token major only)
    FastDiv tok, head, nh; // 16-byte chunks per token, chunks per head, heads
};

// Byte offset within K (or V) of the half's stream byte y < kb.
template <bool FLAT>
__device__ __forceinline__ uint32_t kv_off(const KvStream& s, uint32_t y) {
    if (FLAT) return y;
    const uint32_t c = y >> 4;
    const uint32_t t = fdiv(c, s.tok), r = c - t * s.tok.d;
    const uint32_t bh = fdiv(r, s.head), d = r - bh * s.head.d;
    const uint32_t b = fdiv(bh, s.nh), h = bh - b * s.nh.d;
    return b * s.sB + h * s.sH + t * s.sT + (d << 4) + (y & 15);
}

// Aligned chunks of the stream through K's and V's buffer resources.  The
// resource is chosen per wave (`from`: the wave-uniform lowest and one past
// the highest stream byte its lanes ask for); only a wave across the K/V
// boundary issues both loads, each lane's other one out of range and reading
// nothing.  Chunks past V, and lanes with want false, read as zero.
template <bool FLAT>
struct KvReader {
    const KvStream& s;
    __amdgpu_buffer_rsrc_t rk, rv;
    __device__ __forceinline__ explicit KvReader(const KvStream& st)
        : s(st), rk(chunk_rsrc(st.K, st.ext)), rv(chunk_rsrc(st.V, st.ext)) {}
    struct From {
        bool v, both;
    };
    __device__ __forceinline__ From from(uint32_t lo, uint32_t hi) const {
        return From{lo >= s.kb, lo < s.kb && hi > s.kb};
    }
    __device__ __forceinline__ u32x4 load(uint32_t x, bool want, From f) const {
        const bool in_v = x >= s.kb;
        const uint32_t off = kv_off<FLAT>(s, in_v ? x - s.kb : x);
        const bool ok = want && x < 2 * s.kb;
        u32x4 c = chunk_load(f.v ? rv : rk, ok && in_v == f.v ? off : kNoLoad);
        if (f.both) c |= chunk_load(rv, ok && in_v ? off : kNoLoad);
        return c;
    }
    // the 2-byte word at stream byte x (even), zero past V
    __device__ __forceinline__ uint16_t word(uint32_t x) const {
        if (x >= 2 * s.kb) return 0;
        const bool in_v = x >= s.kb;
        const uint8_t* p = (in_v ? s.V : s.K) + kv_off<FLAT>(s, in_v ? x - s.kb : x);
        return *as_global(reinterpret_cast<const uint16_t*>(p));
    }
};

// The stream chunk at x (x + 16 <= 2 kb, 16-byte aligned), written to K or V.
template <bool FLAT>
__device__ __forceinline__ uint8_t* kv_at(const KvStream& s, uint32_t x) {
    const bool in_v = x >= s.kb;
    return (in_v ? s.V : s.K) + kv_off<FLAT>(s, in_v ? x - s.kb : x);
}

// A whole chunk there.  Non-temporally only where a head is whole 64-byte
// sectors, a line of 128 bytes or more of them: otherwise a sector's bytes come
// from several heads' pieces, and non-temporal stores write it out in parts
// (recovery of 67 MB of K and of V each, 1024 heads: of 16 bytes 165 against 418 us,
// 32 bytes 109 against 245, 48 bytes 95 against 212; 134 MB, 64 heads: 80 bytes half the
// time, 256 bytes 3 to 7 % more).
template <bool FLAT>
__device__ __forceinline__ void kv_put(const KvStream& s, uint32_t x, u32x4 v) {
    uint8_t* p = kv_at<FLAT>(s, x);
    if (!FLAT && ((s.head.d & 3) || s.head.d < 8)) {   // uniform
        // (fenced: the compiler merged the two stores into an ordinary one)
        asm volatile("");
        st16(p, v);
        asm volatile("");
    } else {
        st_stream(p, 0, v);
    }
}

// The byte at stream position x, dropped past V's end.
template <bool FLAT>
__device__ __forceinline__ void kv_put_byte(const KvStream& s, uint32_t x, uint8_t b) {
    if (x < 2 * s.kb) *as_global(kv_at<FLAT>(s, x)) = b;
}

// Bytes of packed row j (Sb bytes each, at sh) that no whole aligned chunk of
// the row holds, b in [0, 32): the at most 15 before the first (b < 16) and
// after the last, copied to K or V.
template <bool FLAT>
__device__ __forceinline__ void kv_put_row_end(const KvStream& s, const uint8_t* sh, uint32_t Sb, uint32_t j,
                                               uint32_t b) {
    const uint32_t r0 = j * Sb, r1 = r0 + Sb, first = (r0 + 15) & ~15u;
    const uint32_t x = b < 16 ? r0 + b : (r1 & ~15u) + (b - 16);
    if (b < 16 ? x < first && x < r1 : x >= first && x < r1) kv_put_byte<FLAT>(s, x, as_global(sh)[x]);
}

// Stream bytes [D0, D0 + nbytes) from the LDS tile (16 bytes of slack) to K
// and V: whole chunks, then the bytes around them.  All BS threads call it.
template <bool FLAT, int BS>
__device__ __forceinline__ void kv_put_tile(const KvStream& s, const uint8_t* tile, uint32_t D0, uint32_t nbytes) {
    const uint32_t out_len = 2 * s.kb;
    const uint32_t E = D0 + nbytes, A0 = (D0 + 15) & ~15u, A1 = E & ~15u;
    auto put_byte = [&](uint32_t x, uint8_t b) {
        if (x < out_len) *as_global(kv_at<FLAT>(s, x)) = b;
    };
    if (A0 < A1) {
        const uint32_t m = A0 - D0;   // < 16
        for (uint32_t k = threadIdx.x; k < (A1 - A0) >> 4; k += BS) {
            u32x4 v = *reinterpret_cast<const u32x4*>(tile + 16 * k);
            if (m) v = funnel16(v, *reinterpret_cast<const u32x4*>(tile + 16 * k + 16), m);
            const uint32_t X = A0 + 16 * k;
            if (X + 16 <= out_len) kv_put<FLAT>(s, X, v);
        }
        const uint32_t i = threadIdx.x;
        if (i < 16 && D0 + i < A0) put_byte(D0 + i, tile[i]);
        else if (i >= 16 && i < 32 && A1 + (i - 16) < E) put_byte(A1 + (i - 16), tile[A1 + (i - 16) - D0]);
    } else {
        for (uint32_t x = D0 + threadIdx.x; x < E; x += BS) put_byte(x, tile[x - D0]);
    }
}

// Host: the stream of K and V indexed [B][H][T][D] with the given byte
// strides.  *flat is set when the token-major order is memory order.  False
// when the layout is not one these kernels take.
struct KvDims {
    int64_t B, H, T, D;        // D in bytes
    int64_t sB, sH, sT;        // byte strides
};
inline bool make_kv_stream(KvStream* s, bool* flat, const void* K, const void* V, KvDims d) {
    if (d.B < 1 || d.H < 1 || d.T < 1 || d.D < 16 || d.D % 16) return false;
    if (!aligned16(K) || !aligned16(V)) return false;
    // a dimension of one element has no stride
    if (d.B == 1) d.sB = 0;
    if (d.H == 1) d.sH = 0;
    if (d.T == 1) d.sT = 0;
    constexpr int64_t lim = int64_t(1) << 31;
    const int64_t st[3] = {d.sB, d.sH, d.sT};
    for (int64_t x : st)
        if (x < 0 || x % 16 || x >= lim) return false;
    if (d.B >= lim || d.H >= lim || d.T >= lim || d.D >= lim) return false;
    const double bytes = double(d.B) * double(d.H) * double(d.T) * double(d.D);
    const double reach = double(d.B - 1) * double(d.sB) + double(d.H - 1) * double(d.sH) +
                         double(d.T - 1) * double(d.sT) + double(d.D);
    if (bytes >= double(1 << 30) || reach >= double(lim)) return false;
    s->K = (uint8_t*)K;
    s->V = (uint8_t*)V;
    s->kb = uint32_t(d.B * d.H * d.T * d.D);
    s->ext = uint32_t((d.B - 1) * d.sB + (d.H - 1) * d.sH + (d.T - 1) * d.sT + d.D);
    s->sB = uint32_t(d.sB);
    s->sH = uint32_t(d.sH);
    s->sT = uint32_t(d.sT);
    s->tok = make_fastdiv(uint32_t(d.B * d.H * d.D / 16));
    s->head = make_fastdiv(uint32_t(d.D / 16));
    s->nh = make_fastdiv(uint32_t(d.H));
    *flat = (d.H == 1 || d.sH == d.D) && (d.B == 1 || d.sB == d.H * d.D) && (d.T == 1 || d.sT == d.B * d.H * d.D);
    return true;
}

}  // namespace kvec
