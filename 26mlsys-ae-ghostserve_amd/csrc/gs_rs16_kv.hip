// gs_rs16_kv.hip -- the wrappers' Reed-Solomon code over GF(2^16)
// (rs.forward_encode_kv, rs.backwards_decode_kv) straight from and to K and V.
//
// The reference packs K || V into a padded tensor and encodes that
// (benchmark/rs/main.py:63-137), and decodes into the shard tensor before it
// splits the rows into K and V (:140-206).  Here one kernel reads K and V and
// writes the data rows and the parity rows, and one reads the surviving rows
// and writes K, V and the rebuilt rows.  The field is that of
// init_gf_tables(): polynomial 0x1100B, generator 2, so the reduction word is
// a constant, and the indices come from the host, which inverts the matrix.
//
// A wave owns NW KiB of every row and walks the rows from the last to the
// first (Horner's rule: parity p = (...(D_{k-1} g + D_{k-2}) g + ...) g + D_0,
// g = 2^(p+1)), each row's chunks loaded two rows ahead.
//
// Products.  With one or two outputs the accumulators hold packed words and
// are doubled in place (gf16.h, about 5 VALU operations per two doublings of
// a dword).  From three outputs on, each thread's 64 bytes of a row are turned
// into sixteen registers, register b holding bit b of its 32 words (a 16 x 16
// bit transposition: four stages of pairwise swaps, 7 operations per dword).
// There a doubling is a renaming of registers and three XORs, the taps of the
// polynomial, so g_p and the next row cost about 17 operations per 16 dwords
// whatever p is: 11 per dword of input for four parities against 28.
//
// Bound by HBM.  Measured (fresh inputs and outputs, one box): RS(6, 2) of 16 x
// 8 x 2048 x 128 bf16, rows off 16-byte alignment, 61 us for 313 MB (5.1 TB/s;
// 57 % of the bytes are writes) against 85 us for pack, zero fill and encode;
// RS(16, 4) of half that stream 28 us for 151 MB (5.3 TB/s) against 47 us.
// Tiles of 2 to 16 KiB, one to four windows a thread, plain or non-temporal
// accesses: 60-65 us and 28-30 us.
#include "gf16.h"
#include "kv_stream.h"

namespace kvec {

constexpr uint16_t kRed = 0x100B;   // x^16 reduced

// ------------------------------------------------------------- bit planes
// r[i] and r[i + s] for every i with bit s clear: swap bit s of the register
// index with bit s of the bit position within each 16-bit word.
template <int s>
__device__ __forceinline__ void plane_swap(uint32_t (&r)[16]) {
    constexpr uint32_t m = s == 8 ? 0x00FF00FFu : s == 4 ? 0x0F0F0F0Fu : s == 2 ? 0x33333333u : 0x55555555u;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        if (i & s) continue;
        const uint32_t a = r[i], b = r[i + s];
        if (s == 8) {
            r[i] = __builtin_amdgcn_perm(b, a, 0x06020400u);
            r[i + s] = __builtin_amdgcn_perm(b, a, 0x07030501u);
        } else {
            // 0xE4: (first & m) | (second & ~m)
            r[i] = __builtin_amdgcn_bitop3_b32(a, b << s, m, 0xE4);
            r[i + s] = __builtin_amdgcn_bitop3_b32(a >> s, b, m, 0xE4);
        }
    }
}

// Computes the sixteen registers here: left free, the compiler interleaved the
// accumulators' steps and held their old and new planes at once.
__device__ __forceinline__ void pin(uint32_t (&r)[16]) {
    asm volatile("" : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]), "+v"(r[4]), "+v"(r[5]), "+v"(r[6]), "+v"(r[7]),
                      "+v"(r[8]), "+v"(r[9]), "+v"(r[10]), "+v"(r[11]), "+v"(r[12]), "+v"(r[13]), "+v"(r[14]),
                      "+v"(r[15]));
    __builtin_amdgcn_sched_barrier(0);
}

// Sixteen dwords of packed words to sixteen bit planes, and back (the swaps
// are their own inverses and commute).
__device__ __forceinline__ void to_planes(uint32_t (&r)[16]) {
    plane_swap<8>(r);
    plane_swap<4>(r);
    plane_swap<2>(r);
    plane_swap<1>(r);
}

// x^(16 + j) reduced
constexpr uint16_t red_pow(int j) {
    uint32_t v = kRed;
    for (int i = 0; i < j; ++i) v = (v << 1) ^ ((v & 0x8000u) ? 0x10000u | kRed : 0u);
    return uint16_t(v);
}

// a = a * 2^E ^ d on bit planes (d null: no addend).  Plane i of the product
// is plane i - E of a and, for each of the E planes shifted out, that plane
// where x^(16 + j) reduced has bit i.
template <int E, bool ADD>
__device__ __forceinline__ void plane_step(uint32_t (&a)[16], const uint32_t (&d)[16]) {
    uint32_t out[16];
#pragma unroll
    for (int i = 15; i >= 0; --i) {
        uint32_t t[E + 2];
        int n = 0;
        if (ADD) t[n++] = d[i];
        if (i >= E) t[n++] = a[i >= E ? i - E : 0];
#pragma unroll
        for (int j = 0; j < E; ++j)
            if ((red_pow(j) >> i) & 1) t[n++] = a[16 - E + j];
        uint32_t v = n == 0 ? 0u : t[0];
        int q = 1;
#pragma unroll
        for (; q + 1 < n; q += 2) v = xor3(v, t[q], t[q + 1]);
        if (q < n) v ^= t[q];
        out[i] = v;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) a[i] = out[i];
}

// -------------------------------------------------------------- accumulators
// Outputs p = 0 .. M-1 with multipliers 2^(p+1).
template <int M, int NW, bool PLANES>
struct RsAcc;

template <int M>
struct RsAcc<M, 4, true> {
    uint32_t a[M][16];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int p = 0; p < M; ++p)
#pragma unroll
            for (int i = 0; i < 16; ++i) a[p][i] = 0;
    }
    template <int P = 0>
    __device__ __forceinline__ void add(const uint32_t (&d)[16]) {
        if constexpr (P < M) {
            plane_step<P + 1, true>(a[P], d);
            pin(a[P]);
            add<P + 1>(d);
        }
    }
    template <int P = 0>
    __device__ __forceinline__ void shift() {
        if constexpr (P < M) {
            plane_step<P + 1, false>(a[P], a[P]);
            shift<P + 1>();
        }
    }
    // every accumulator times its multiplier, plus the row's windows
    __device__ __forceinline__ void fold(const u32x4 (&x)[4]) {
        uint32_t d[16];
#pragma unroll
        for (int n = 0; n < 4; ++n) d[4 * n] = x[n].x, d[4 * n + 1] = x[n].y, d[4 * n + 2] = x[n].z, d[4 * n + 3] = x[n].w;
        to_planes(d);
        pin(d);
        add(d);
    }
    __device__ __forceinline__ void finish() {
#pragma unroll
        for (int p = 0; p < M; ++p) to_planes(a[p]);
    }
    __device__ __forceinline__ u32x4 window(int p, int n) const {
        return u32x4{a[p][4 * n], a[p][4 * n + 1], a[p][4 * n + 2], a[p][4 * n + 3]};
    }
};

template <int M, int NW>
struct RsAcc<M, NW, false> {
    static_assert(M <= 2, "packed words: one or two outputs");
    uint32_t a[M][NW][4];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int p = 0; p < M; ++p)
#pragma unroll
            for (int n = 0; n < NW; ++n) a[p][n][0] = a[p][n][1] = a[p][n][2] = a[p][n][3] = 0;
    }
    __device__ __forceinline__ void step(const u32x4* x) {
        constexpr Gf16Quad quad = {uint32_t(kRed) << 16,
                                   uint32_t(red_pow(1)) | (uint32_t(uint16_t(kRed ^ red_pow(1))) << 16)};
#pragma unroll
        for (int n = 0; n < NW; ++n) {
            const uint32_t y[4] = {x ? x[n].x : 0u, x ? x[n].y : 0u, x ? x[n].z : 0u, x ? x[n].w : 0u};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                a[0][n][q] = gf16_dbl2_xor(a[0][n][q], uint32_t(kRed) * 0x10001u, y[q]);
                if (M > 1) a[M - 1][n][q] = gf16_quad2_xor(a[M - 1][n][q], quad, y[q]);
            }
        }
    }
    __device__ __forceinline__ void fold(const u32x4 (&x)[NW]) { step(x); }
    __device__ __forceinline__ void shift() { step(nullptr); }
    __device__ __forceinline__ void finish() {}
    __device__ __forceinline__ u32x4 window(int p, int n) const {
        return u32x4{a[p][n][0], a[p][n][1], a[p][n][2], a[p][n][3]};
    }
};

// The wave's NW consecutive KiB of one row: aligned chunks, and lane 63's
// chunk after the last (rows at other than 16-byte alignments).
template <int NW, bool ALIGNED>
struct RowChunks {
    u32x4 c[NW], e;
    // the windows, m bytes into the chunks (wave-uniform)
    __device__ __forceinline__ void windows(uint32_t m, u32x4 (&x)[NW]) const {
#pragma unroll
        for (int n = 0; n < NW; ++n) x[n] = c[n];
        if (ALIGNED || m == 0) return;
#pragma unroll
        for (int n = 0; n < NW; ++n) {
            u32x4 next = e;
            if (n + 1 < NW) {
                const u32x4 f = c[n + 1 < NW ? n + 1 : n];
                auto lane0 = [](uint32_t v) { return uint32_t(__builtin_amdgcn_readfirstlane(int(v))); };
                next = u32x4{lane0(f.x), lane0(f.y), lane0(f.z), lane0(f.w)};
            }
            x[n] = funnel16(c[n], from_next_lane_or(c[n], next), m);
        }
    }
};

// ------------------------------------------------------------------- encode
// k data rows (the stream K || V || zeros cut into rows of Sb bytes) and M
// parity rows of the shard tensor sh, from K and V.  ALIGNED: Sb is a multiple
// of 16, so windows are chunks and the parities go out from registers.
template <int M, int NW, bool PLANES, int BS, bool ALIGNED>
__global__ __launch_bounds__(BS) void rs16_encode_kv_kernel(KvStream src, uint8_t* sh, uint32_t Sb, int k) {
    constexpr uint32_t TB = 16 * BS * NW, WB = 1024 * NW;
    __shared__ __attribute__((aligned(16))) uint8_t tile[ALIGNED ? 1 : M][ALIGNED ? 16 : TB + 16];
    const uint32_t t0 = blockIdx.x * TB;
    const uint32_t nbytes = Sb - t0 < TB ? Sb - t0 : TB;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wb = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6))) * WB;
    const uint32_t data_end = uint32_t(k) * Sb;
    const uint32_t kb = src.kb;
    auto at = [&](int i) { return uint32_t(i) * Sb + t0 + wb; };
    auto load = [&](int i, RowChunks<NW, ALIGNED>& s) {
        if (i < 0) return;   // uniform
        const uint32_t A = at(i), m = ALIGNED ? 0 : A & 15, x = A - m, end = x + WB + (ALIGNED ? 0 : 16);
        const bool in_v = x >= kb;
        if (end <= kb || (in_v && end <= 2 * kb)) {   // uniform: one piece of K or of V
            const uint8_t* p = in_v ? src.V + (x - kb) : src.K + x;
#pragma unroll
            for (int n = 0; n < NW; ++n) s.c[n] = ld_stream(p + n * 1024, 16 * lane);
            if (!ALIGNED) s.e = ld16(p + WB);
        } else {   // chunks past V's end read its last one; mask() clears them
            auto chunk = [&](uint32_t y) {
                y = y < 2 * kb - 16 ? y : 2 * kb - 16;
                return ld16(y >= kb ? src.V + (y - kb) : src.K + y);
            };
#pragma unroll
            for (int n = 0; n < NW; ++n) s.c[n] = chunk(x + n * 1024 + 16 * lane);
            if (!ALIGNED) s.e = chunk(x + WB);
        }
    };
    RsAcc<M, NW, PLANES> acc;
    acc.clear();
    auto use = [&](int i, RowChunks<NW, ALIGNED>& s) {
        const uint32_t A = at(i), m = ALIGNED ? 0 : A & 15, x = A - m, rend = uint32_t(i + 1) * Sb;
        if (x + WB + 16 > 2 * kb) {   // uniform
            const u32x4 zero = {0, 0, 0, 0};
#pragma unroll
            for (int n = 0; n < NW; ++n)
                if (x + n * 1024 + 16 * lane >= 2 * kb) s.c[n] = zero;
            if (!ALIGNED && x + WB >= 2 * kb) s.e = zero;
        }
        // the chunks into the data rows: non-temporal, except in the two
        // 128-byte lines shared with the neighbouring waves; the last data
        // row's partial last chunk is written below
        const uint32_t pre = ((uint32_t(reinterpret_cast<uintptr_t>(sh)) + x) >> 4) & 7;
#pragma unroll
        for (int n = 0; n < NW; ++n) {
            const uint32_t X = x + n * 1024 + 16 * lane;
            if (X < rend && X + 16 <= data_end) {
                const bool shared = pre != 0 && ((n == 0 && lane < 8 - pre) || (n == NW - 1 && lane >= 64 - pre));
                if (shared) st16(sh + X, s.c[n]);
                else st_stream(sh, X, s.c[n]);
            }
        }
        // a row that ends with the tile can end in the chunk after it
        if (!ALIGNED && m && wb + WB == TB && t0 + TB >= Sb && lane == 63 && x + WB < rend && x + WB + 16 <= data_end)
            st16(sh + x + WB, s.e);
        u32x4 w[NW];
        s.windows(m, w);
        acc.fold(w);
    };
    if (!ALIGNED && t0 + TB >= Sb && threadIdx.x < 8) {
        const uint32_t X = (data_end & ~15u) + 2 * threadIdx.x;
        if (X < data_end) *as_global(reinterpret_cast<uint16_t*>(sh + X)) = KvReader<true>(src).word(X);
    }
    // Two sets, the loop unrolled by two so that none is copied; an odd k gets
    // a row of zeros above the last, which leaves the accumulators zero.
    RowChunks<NW, ALIGNED> ra, rb;
    int i = (k - 1) | 1;
    load(i, ra);
    load(i - 1, rb);
    for (; i > 0; i -= 2) {
        use(i, ra);
        load(i - 2, ra);
        use(i - 1, rb);
        load(i - 3, rb);
    }
    acc.finish();
    uint8_t* par = sh + data_end + t0;
#pragma unroll
    for (int p = 0; p < M; ++p)
#pragma unroll
        for (int n = 0; n < NW; ++n) {
            const uint32_t o = wb + n * 1024 + 16 * lane;
            if (!ALIGNED) *reinterpret_cast<u32x4*>(tile[p] + o) = acc.window(p, n);
            else if (o < nbytes) st_stream(par + uint32_t(p) * Sb, o, acc.window(p, n));
        }
    if (ALIGNED) return;
    __syncthreads();
#pragma unroll
    for (int p = 0; p < M; ++p) tile_store<true, BS>(par + uint32_t(p) * Sb, tile[p], nbytes);
}

// ---------------------------------------------------------------- host side
typedef void (*RsEncKvFn)(KvStream, uint8_t*, uint32_t, int);
struct RsKvKern {
    RsEncKvFn fn;
    int bs, nw;
};

template <bool ALIGNED>
static RsKvKern rs_encode_kv(int m) {
    switch (m) {
        case 1: return {&rs16_encode_kv_kernel<1, 2, false, 256, ALIGNED>, 256, 2};
        case 2: return {&rs16_encode_kv_kernel<2, 2, false, 256, ALIGNED>, 256, 2};
        case 3: return {&rs16_encode_kv_kernel<3, 4, true, 256, ALIGNED>, 256, 4};
        case 4: return {&rs16_encode_kv_kernel<4, 4, true, 256, ALIGNED>, 256, 4};
        default: return {nullptr, 0, 0};
    }
}

}  // namespace kvec

using namespace kvec;

extern "C" int kvec_rs16_encode_kv(const void* key_input, const void* value_input, int64_t kv_half_bytes, void* shards,
                                   int data_shards, int parity_shards, int shard_size, void* stream) {
    static const char* fn = "kvec_rs16_encode_kv";
    if (!shards) return set_error(KVEC_EINVAL, "%s: null pointer", fn);
    KvStream s{};
    bool flat = false;
    const uint64_t Sb = uint64_t(shard_size > 0 ? shard_size : 0) * 2;
    const RsKvKern kern = Sb % 16 == 0 ? rs_encode_kv<true>(parity_shards) : rs_encode_kv<false>(parity_shards);
    const uint64_t rows = uint64_t(data_shards > 0 ? data_shards : 0) + uint64_t(parity_shards > 0 ? parity_shards : 0);
    if (!kern.fn || data_shards < 1 || data_shards > 65535 || shard_size < 64 || !aligned16(shards) ||
        rows * Sb > (uint64_t(1) << 31) - 16 || kv_half_bytes < 16 ||
        !make_kv_stream(&s, &flat, key_input, value_input, KvDims{1, 1, 1, kv_half_bytes, 0, 0, 0}) ||
        2 * uint64_t(s.kb) > uint64_t(data_shards) * Sb)
        return set_error(KVEC_EUNSUPPORTED, "%s: layout or stripe not built", fn);
    if (!key_input || !value_input) return set_error(KVEC_EINVAL, "%s: null K or V", fn);
    const Span w = {shards, rows * Sb, "shards", -1};
    const Span r[2] = {{key_input, s.kb, "K", -1}, {value_input, s.kb, "V", -1}};
    if (int rc = check_no_alias(&w, 1, r, 2, fn)) return rc;
    hipLaunchKernelGGL(kern.fn, dim3(blocks_for(int64_t(Sb), 16 * kern.bs * kern.nw)), dim3(kern.bs), 0,
                       as_stream(stream), s, (uint8_t*)shards, uint32_t(Sb), data_shards);
    return check_launch(fn);
}
