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
// g = 2^(p+1)), each row's chunks loaded two or four rows ahead.
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
            pin(a[P]);
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
    // after finish()
    __device__ __forceinline__ void add_window(int p, int n, u32x4 v) {
        a[p][4 * n] ^= v.x, a[p][4 * n + 1] ^= v.y, a[p][4 * n + 2] ^= v.z, a[p][4 * n + 3] ^= v.w;
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
    __device__ __forceinline__ void add_window(int p, int n, u32x4 v) {
        a[p][n][0] ^= v.x, a[p][n][1] ^= v.y, a[p][n][2] ^= v.z, a[p][n][3] ^= v.w;
    }
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
    // Two sets, the loop unrolled by two so that none is copied; the last row
    // of an odd k comes before it (a skip inside cost 16 % in copies).
    RowChunks<NW, ALIGNED> ra, rb;
    int i = k - 1;
    if (k & 1) {
        load(i, rb);
        load(i - 1, ra);
        use(i, rb);
        load(i - 2, rb);
        --i;
    } else {
        load(i, ra);
        load(i - 1, rb);
    }
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

// ------------------------------------------------------------------- decode
// M lost data rows of a shard tensor sh from the surviving rows and parity
// rows 0 .. M-1: syndrome r is b_r = Par_r ^ XOR_j D_j 2^((r+1) j) over the
// surviving rows, by Horner's rule over all k rows with a lost row adding
// nothing, and the lost rows are x_c = XOR_r inv[c][r] b_r through byte maps
// (gf16.h) that the host built and each block stages in LDS.  The surviving
// rows' whole chunks go to K and V from the registers they were loaded into,
// their ends byte by byte from block 0, the rebuilt rows to their place in sh
// and to K and V.
// Measured (kernel trace, fresh outputs): two of six rows lost, 16 x 8 x 2048
// x 128 bf16, 57 us for 313 MB (5.5 TB/s); 4 x 8 x 1001 x 128 13.7 us for 38 MB,
// where the reconstruct and the copies took 19 us beside two blocking uploads
// of the indices (whole call 60 -> 14 us).
template <int M>
struct RsRec {
    uint64_t lost;        // data rows, bit i
    uint32_t row[M];      // the lost rows, in order
    uint32_t maps[M * M][kRs16Tab];
};

template <int M, int NW, int R, bool PLANES, int BS, bool ALIGNED>
__global__ __launch_bounds__(BS) void rs16_recover_kv_kernel(KvStream dst, uint8_t* sh, uint32_t sh_bytes, uint32_t Sb,
                                                             int k, RsRec<M> rec) {
    constexpr uint32_t TB = 16 * BS * NW, WB = 1024 * NW;
    __shared__ __attribute__((aligned(16))) uint8_t tile[ALIGNED ? 1 : M][ALIGNED ? 16 : TB + 16];
    __shared__ __attribute__((aligned(16))) uint32_t maps[M * M][kRs16Tab];
    for (uint32_t e = threadIdx.x; e < M * M * kRs16Tab; e += BS) maps[e / kRs16Tab][e % kRs16Tab] = rec.maps[e / kRs16Tab][e % kRs16Tab];
    const uint32_t t0 = blockIdx.x * TB;
    const uint32_t nbytes = Sb - t0 < TB ? Sb - t0 : TB;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wb = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6))) * WB;
    const uint32_t kb = dst.kb;
    const __amdgpu_buffer_rsrc_t rs = chunk_rsrc(sh, (sh_bytes + 15) & ~15u);
    auto absent = [&](int i) { return i >= k || ((rec.lost >> (i & 63)) & 1); };   // i >= 0
    auto at = [&](int i) { return uint32_t(i >= 0 ? i : k - 1 - i) * Sb + t0 + wb; };
    // row i, or parity row -1 - i
    auto load = [&](int i, RowChunks<NW, ALIGNED>& s) {
        if (i < -M || (i >= 0 && absent(i))) return;   // uniform
        const uint32_t A = at(i), m = ALIGNED ? 0 : A & 15, x = A - m;
#pragma unroll
        for (int n = 0; n < NW; ++n) s.c[n] = chunk_load(rs, x + n * 1024 + 16 * lane);
        if (!ALIGNED) s.e = chunk_load(rs, x + WB);
    };
    RsAcc<M, NW, PLANES> acc;
    acc.clear();
    auto use = [&](int i, const RowChunks<NW, ALIGNED>& s) {
        if (!PLANES && i >= k) return;   // the accumulators are still zero
        if (absent(i)) {
            acc.shift();
            return;
        }
        const uint32_t A = at(i), m = ALIGNED ? 0 : A & 15, x = A - m, r0 = uint32_t(i) * Sb, rend = r0 + Sb;
        if (x >= r0 && x + WB <= rend && (x + WB <= kb || (x >= kb && x + WB <= 2 * kb))) {   // uniform
            uint8_t* p = x >= kb ? dst.V + (x - kb) : dst.K + x;
#pragma unroll
            for (int n = 0; n < NW; ++n) st_stream(p + n * 1024, 16 * lane, s.c[n]);
        } else {
#pragma unroll
            for (int n = 0; n < NW; ++n) {
                const uint32_t X = x + n * 1024 + 16 * lane;
                if (X >= r0 && X + 16 <= rend && X < 2 * kb) st_stream(kv_at<true>(dst, X), 0, s.c[n]);
            }
        }
        u32x4 w[NW];
        s.windows(m, w);
        acc.fold(w);
    };
    if (!ALIGNED && blockIdx.x == 0)
        for (uint32_t u = threadIdx.x; u < 32 * uint32_t(k); u += BS)
            if (!absent(int(u >> 5))) kv_put_row_end<true>(dst, sh, Sb, u >> 5, u & 31);
    RowChunks<NW, ALIGNED> row[R];
    int i = (k + R - 1) / R * R - 1;
#pragma unroll
    for (int j = 0; j < R; ++j) load(i - j, row[j]);
    for (; i >= 0; i -= R) {
#pragma unroll
        for (int j = 0; j < R; ++j) {
            use(i - j, row[j]);
            load(i - j - R, row[j]);
        }
    }
    // row[r] holds parity row r
    acc.finish();
#pragma unroll
    for (int r = 0; r < M; ++r) {
        u32x4 w[NW];
        row[r % R].windows(ALIGNED ? 0 : at(-1 - r) & 15, w);
#pragma unroll
        for (int n = 0; n < NW; ++n) acc.add_window(r, n, w[n]);
        if (r + R < M) load(-1 - r - R, row[r % R]);
    }
    __syncthreads();   // maps
#pragma unroll
    for (int n = 0; n < NW; ++n) {
        Gf8Fields f[M][4];
#pragma unroll
        for (int r = 0; r < M; ++r) {
            uint32_t by[4];
            split_bytes(acc.window(r, n), by);
#pragma unroll
            for (int q = 0; q < 4; ++q) f[r][q] = gf8_fields(by[q]);
        }
        const uint32_t o = wb + n * 1024 + 16 * lane;
#pragma unroll
        for (int c = 0; c < M; ++c) {
            uint32_t v[4] = {0, 0, 0, 0};
#pragma unroll
            for (int r = 0; r < M; ++r) {
                const uint32_t* T = maps[c * M + r];
                v[0] = gf16_fma2(v[0], f[r][0], T + 0, f[r][1], T + 6);
                v[1] = gf16_fma2(v[1], f[r][0], T + 12, f[r][1], T + 18);
                v[2] = gf16_fma2(v[2], f[r][2], T + 0, f[r][3], T + 6);
                v[3] = gf16_fma2(v[3], f[r][2], T + 12, f[r][3], T + 18);
                // one coefficient's maps live at a time
                asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]) :: "memory");
                __builtin_amdgcn_sched_barrier(0);
            }
            const u32x4 x = join_bytes(v);
            if (!ALIGNED) {
                *reinterpret_cast<u32x4*>(tile[c] + o) = x;
            } else if (o < nbytes) {
                const uint32_t X = rec.row[c] * Sb + t0 + o;
                st_stream(sh, X, x);
                if (X < 2 * kb) st_stream(kv_at<true>(dst, X), 0, x);
            }
        }
    }
    if (ALIGNED) return;
    __syncthreads();
#pragma unroll
    for (int c = 0; c < M; ++c) {
        tile_store<false, BS>(sh + rec.row[c] * Sb + t0, tile[c], nbytes);
        kv_put_tile<true, BS>(dst, tile[c], rec.row[c] * Sb + t0, nbytes);
    }
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

// ------------------------------------------------ the inverse, on the host
struct Gf16Tables {
    uint16_t ex[2 * 65535], lg[65536];
    Gf16Tables() { kvec_gf16_tables(ex, lg); }
    uint16_t mul(uint16_t a, uint16_t b) const { return a && b ? ex[uint32_t(lg[a]) + lg[b]] : uint16_t(0); }
    uint16_t inv(uint16_t a) const { return ex[65535 - lg[a]]; }   // a != 0
};

static const Gf16Tables& gf16_tables() {
    static const Gf16Tables t;
    return t;
}

// Inverse of V[r][c] = 2^((r + 1) row[c]) by the reference's Gauss-Jordan
// (benchmark/rs/kernel.cu:135-185: pivot order, a zero column skipped).
template <int M>
static void rs_inverse(const uint32_t* row, uint16_t (&inv)[M][M]) {
    const Gf16Tables& g = gf16_tables();
    uint16_t V[M][M];
    for (int r = 0; r < M; ++r)
        for (int c = 0; c < M; ++c) {
            V[r][c] = g.ex[(uint32_t(r + 1) * row[c]) % 65535];
            inv[r][c] = r == c;
        }
    for (int i = 0; i < M; ++i) {
        int pr = i;
        while (pr < M && V[pr][i] == 0) ++pr;
        if (pr == M) continue;
        for (int c = 0; c < M && pr != i; ++c) {
            uint16_t t = V[i][c];
            V[i][c] = V[pr][c], V[pr][c] = t;
            t = inv[i][c];
            inv[i][c] = inv[pr][c], inv[pr][c] = t;
        }
        const uint16_t ip = g.inv(V[i][i]);
        for (int c = 0; c < M; ++c) {
            V[i][c] = g.mul(V[i][c], ip);
            inv[i][c] = g.mul(inv[i][c], ip);
        }
        for (int r = 0; r < M; ++r) {
            const uint16_t f = V[r][i];
            if (r == i || !f) continue;
            for (int c = 0; c < M; ++c) {
                V[r][c] ^= g.mul(f, V[i][c]);
                inv[r][c] ^= g.mul(f, inv[i][c]);
            }
        }
    }
}

// The byte maps of coefficient c in the order gf16_fma2 reads them: low to
// low, high to low, low to high, high to high byte; two dwords per 3-bit field.
static void byte_maps(uint16_t c, uint32_t (&out)[kRs16Tab]) {
    const Gf16Tables& g = gf16_tables();
    for (int d = 0; d < kRs16Tab; ++d) {
        const int src = (d / 6) & 1, dst = d / 12, f = (d % 6) >> 1, half = d & 1;
        uint32_t dw = 0;
        for (int q = 0; q < 4; ++q) {
            const int v = half * 4 + q;
            if (f == 2 && v >= 4) continue;
            const uint16_t y = g.mul(uint16_t((v << (3 * f)) << (8 * src)), c);
            dw |= uint32_t((y >> (8 * dst)) & 0xFF) << (8 * q);
        }
        out[d] = dw;
    }
}

// One or two lost rows: 256 threads with four rows in flight, or 512 with two
// from 8 MiB rows on.  Whole calls, 256 threads against 512: RS(4, 1) rows of 2 to
// 7 MB 11.3-11.6 against 11.9-13.1 us, 9 MB 16.3 against 16.8, 22 MB 34.8 against
// 33.9; RS(6, 2) 2 MB 12.6 against 13.1, 9 MB 25.6 against 26.6, 22 MB 56.9 against
// 56.1; RS(10, 2) 30 MB 122.6 against 119.2.  They cross between 10 and 12 MB, so
// rows of 8 to 11 MB give away up to 4 %.  More lost rows: bit planes, two rows of
// four windows in flight; 128 and 512 threads ran 39 and 43 against 35 us (16 rows
// of 4.2 MB, four lost).
template <int M>
static void rs_recover_launch(KvStream dst, uint8_t* sh, uint64_t sh_bytes, uint32_t Sb, int k, const int32_t* missing,
                              hipStream_t st) {
    RsRec<M> rec{};
    for (int c = 0; c < M; ++c) {
        rec.row[c] = uint32_t(missing[c]);
        rec.lost |= uint64_t(1) << missing[c];
    }
    uint16_t inv[M][M];
    rs_inverse<M>(rec.row, inv);
    for (int c = 0; c < M; ++c)
        for (int r = 0; r < M; ++r) byte_maps(inv[c][r], rec.maps[c * M + r]);
    auto launch = [&](auto kern, int bs, int nw) {
        hipLaunchKernelGGL(kern, dim3(blocks_for(int64_t(Sb), 16 * bs * nw)), dim3(bs), 0, st, dst, sh,
                           uint32_t(sh_bytes), Sb, k, rec);
    };
    const bool aligned = Sb % 16 == 0;
    if constexpr (M > 2) {
        if (aligned) launch(&rs16_recover_kv_kernel<M, 4, 2, true, 256, true>, 256, 4);
        else launch(&rs16_recover_kv_kernel<M, 4, 2, true, 256, false>, 256, 4);
    } else if (Sb < (8u << 20)) {
        if (aligned) launch(&rs16_recover_kv_kernel<M, 1, 4, false, 256, true>, 256, 1);
        else launch(&rs16_recover_kv_kernel<M, 1, 4, false, 256, false>, 256, 1);
    } else {
        if (aligned) launch(&rs16_recover_kv_kernel<M, 1, 2, false, 512, true>, 512, 1);
        else launch(&rs16_recover_kv_kernel<M, 1, 2, false, 512, false>, 512, 1);
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
        2 * uint64_t(s.kb) > uint64_t(data_shards) * Sb || rs16_ring_encode_faster(data_shards, parity_shards, Sb))
        return set_error(KVEC_EUNSUPPORTED, "%s: layout or stripe not built", fn);
    if (!key_input || !value_input) return set_error(KVEC_EINVAL, "%s: null K or V", fn);
    const Span w = {shards, rows * Sb, "shards", -1};
    const Span r[2] = {{key_input, s.kb, "K", -1}, {value_input, s.kb, "V", -1}};
    if (int rc = check_no_alias(&w, 1, r, 2, fn)) return rc;
    hipLaunchKernelGGL(kern.fn, dim3(blocks_for(int64_t(Sb), 16 * kern.bs * kern.nw)), dim3(kern.bs), 0,
                       as_stream(stream), s, (uint8_t*)shards, uint32_t(Sb), data_shards);
    return check_launch(fn);
}

extern "C" int kvec_rs16_recover_kv(void* shards, void* key_output, void* value_output, int64_t kv_half_bytes,
                                    int data_shards, int parity_shards, int shard_size, const int32_t* missing,
                                    int n_missing, void* stream) {
    static const char* fn = "kvec_rs16_recover_kv";
    if (!shards || (n_missing > 0 && !missing)) return set_error(KVEC_EINVAL, "%s: null pointer", fn);
    if (n_missing > 0 && n_missing > parity_shards)
        return set_error(KVEC_EINVAL, "%s: %d lost rows, %d parity rows", fn, n_missing, parity_shards);
    for (int q = 0; q < n_missing; ++q)
        if (missing[q] < 0 || missing[q] >= data_shards || (q && missing[q] <= missing[q - 1]))
            return set_error(KVEC_EINVAL, "%s: lost rows must be ascending data rows", fn);
    KvStream s{};
    bool flat = false;
    const uint64_t Sb = uint64_t(shard_size > 0 ? shard_size : 0) * 2;
    const uint64_t bytes = Sb * (uint64_t(data_shards > 0 ? data_shards : 0) + uint64_t(parity_shards > 0 ? parity_shards : 0));
    if (n_missing < 1 || n_missing > 4 || data_shards < 1 || data_shards > 64 || parity_shards > 65535 ||
        shard_size < 64 || !aligned16(shards) || bytes > (uint64_t(1) << 31) - 16 || kv_half_bytes < 16 ||
        !make_kv_stream(&s, &flat, key_output, value_output, KvDims{1, 1, 1, kv_half_bytes, 0, 0, 0}) ||
        2 * uint64_t(s.kb) > uint64_t(data_shards) * Sb)
        return set_error(KVEC_EUNSUPPORTED, "%s: layout or stripe not built", fn);
    if (!key_output || !value_output) return set_error(KVEC_EINVAL, "%s: null K or V", fn);
    const Span w[3] = {{shards, bytes, "shards", -1}, {key_output, s.kb, "K", -1}, {value_output, s.kb, "V", -1}};
    if (int rc = check_no_alias(w, 3, nullptr, 0, fn)) return rc;
    uint8_t* sh = (uint8_t*)shards;
    const hipStream_t st = as_stream(stream);
    switch (n_missing) {
        case 1: rs_recover_launch<1>(s, sh, bytes, uint32_t(Sb), data_shards, missing, st); break;
        case 2: rs_recover_launch<2>(s, sh, bytes, uint32_t(Sb), data_shards, missing, st); break;
        case 3: rs_recover_launch<3>(s, sh, bytes, uint32_t(Sb), data_shards, missing, st); break;
        default: rs_recover_launch<4>(s, sh, bytes, uint32_t(Sb), data_shards, missing, st); break;
    }
    return check_launch(fn);
}
