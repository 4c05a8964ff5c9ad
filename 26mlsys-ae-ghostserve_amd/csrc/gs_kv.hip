// gs_kv.hip -- the star-diagonal code's backup and recovery straight from and
// to K and V tensors indexed [B][H][T][D].
//
// The reference's wrappers permute K and V to token-major copies, pack those
// into the rows and code the rows (benchmark/rdp/main.py:44-92); recovery
// copies the rows out and permutes back (:95-126).  Here the coding kernels
// address the token-major stream in K and V (kv_stream.h), so each byte of K
// and V crosses HBM once.  Bound by HBM: 16 requests x 8 heads x 2047 tokens x
// 128 (bf16, six data rows), kernel trace: backup 56 us (5.6 TB/s of the 313
// MB it must move), recovery 58 us (5.0 TB/s of 291 MB; a wave's 1 KiB of
// stream is four heads, so its stores to K and V are four 256-byte pieces),
// where the torch permutes alone took 99 us beside a 53 us coding kernel.
// Whole calls, A/B: recovery 169 -> 84 us, the reference demo's backup (1 x 8
// x 512 x 128, eight rows) 48 -> 32 us.
#include "gs_star.h"
#include "kv_stream.h"

namespace kvec {

// ------------------------------------------------------------------- backup
// One tile of 16 BS bytes of every row: the ND data rows are the stream
// K || V || zeros laid end to end, row r at stream byte r Sb, and each lane
// loads the aligned stream chunk under its window of every row, all requested
// at once.  It stores the chunk into the data rows (the rows start 16-byte
// aligned, so a stream chunk is a row chunk) and takes the P window (mr bytes
// into the chunk) and the Q window (2 r bytes before that) from it and its
// neighbours' chunks by DPP shifts: with ND <= 8 the Q window starts at most
// 14 bytes before the chunk, with ND <= 16 at most 30.  Lane 63 loads the chunk
// after the wave's and lane 0 the one before it into one register set, the edge
// value of both shifts; rows past 8 have one more for the second chunk before.
// P and Q go through LDS to tile_store.
// Q words 0 .. ND-2 wrap: block 0's first threads compute each from its ND
// words, requested before the rows, and they replace what the shifts gave.
// kRows: the rows are in place already, at any word alignment; nothing but P
// and Q is written.  For nine rows and more, which the packed kernel takes one
// at a time: 16 rows of 1 MB 64.6 -> 7.4 us (kernel trace), and the backup of
// ten rows from K and V (33 MB) 55 -> 13 us beside 23 us less of permutes.
enum PqSource { kRows, kFlat, kTokens };

template <int ND, int BS, PqSource SRC>
__global__ __launch_bounds__(BS) void gs_backup_kv_kernel(KvStream src, uint8_t* sh, uint32_t Sb, GsStar star) {
    constexpr uint32_t TB = 16 * BS;
    constexpr bool ROWS = SRC == kRows;
    __shared__ __attribute__((aligned(16))) uint8_t tp[TB + 16];
    __shared__ __attribute__((aligned(16))) uint8_t tq[TB + 16];
    const uint32_t t0 = blockIdx.x * TB;
    const uint32_t nbytes = Sb - t0 < TB ? Sb - t0 : TB;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t w64 = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6))) * 1024;
    const uint32_t data_end = uint32_t(ND) * Sb;
    // the rows start b15 bytes past the 16-byte boundary that offsets count from
    const uint32_t b15 = ROWS ? uint32_t(reinterpret_cast<uintptr_t>(sh)) & 15 : 0;
    const KvReader<SRC == kFlat> in(src);
    const __amdgpu_buffer_rsrc_t rrows = chunk_rsrc(sh - b15, (b15 + uint32_t(ND + 2) * Sb + 15) & ~15u);
    auto load = [&](uint32_t x, bool want, typename KvReader<SRC == kFlat>::From f) {
        if constexpr (ROWS) return chunk_load(rrows, want ? x : kNoLoad);
        else return in.load(x, want, f);
    };
    auto row_m = [&](int r) { return (b15 + uint32_t(r) * Sb + t0) & 15; };
    auto row_x0 = [&](int r) { return b15 + uint32_t(r) * Sb + t0 - row_m(r); };
    // wrapped Q words
    const bool wraps = ND > 1 && t0 == 0 && threadIdx.x < ND - 1;
    uint16_t wq[ND];
    if (wraps) {
        const uint32_t d = threadIdx.x, S = Sb / 2;
#pragma unroll
        for (int r = 0; r < ND; ++r) {
            const uint32_t w = uint32_t(r) * S + (d >= uint32_t(r) ? d - r : S + d - r);
            wq[r] = ROWS ? as_global(reinterpret_cast<const uint16_t*>(sh))[w] : in.word(2 * w);
        }
    }
    // lanes whose chunk holds no byte any window of the row uses load nothing
    const bool live = 16 * threadIdx.x < nbytes + 16;
    constexpr int NE = ND > 8 ? ND - 8 : 1;
    u32x4 c0[ND], e[ND], e2[NE];
#pragma unroll
    for (int r = 0; r < ND; ++r) {
        const uint32_t mr = row_m(r), x0 = row_x0(r), X = x0 + 16 * threadIdx.x;
        const int s = int(mr) - 2 * r;
        const uint32_t lo = x0 + w64;   // the wave's chunks, and one or two before and one after
        constexpr uint32_t back = ND > 8 ? 32 : 16;
        const auto f = in.from(lo >= back ? lo - back : 0, lo + 1024 + 16);
        c0[r] = load(X, live, f);
        const bool want = (lane == 63 && (mr > 0 || s > 0)) || (lane == 0 && s < 0 && X != 0);
        e[r] = load(lane == 63 ? X + 16 : X - 16, live && want, f);
        if (r >= 8) e2[r >= 8 ? r - 8 : 0] = load(X - 32, live && lane == 0 && s < -16, f);
    }
    __builtin_amdgcn_sched_barrier(0);
    const int32_t w0 = int32_t((t0 >> 1) + 8 * threadIdx.x);
    u32x4 p = {0, 0, 0, 0}, q = {0, 0, 0, 0};
#pragma unroll
    for (int r = 0; r < ND; ++r) {
        const uint32_t mr = row_m(r), x0 = row_x0(r), X = x0 + 16 * threadIdx.x;
        const int s = int(mr) - 2 * r;
        const u32x4 c1 = from_next_lane_or(c0[r], e[r]), cm = from_prev_lane_or(c0[r], e[r]);
        if constexpr (!ROWS) {
            // The chunk into the data rows: non-temporal, except in the two
            // 128-byte lines the wave shares with its neighbours (copy_chunk_split).
            // In the row's last tile the last thread also stores the chunk after its
            // own, which a row ending with the tile can end in.
            const uint32_t rend = uint32_t(r + 1) * Sb;
            const uint32_t pre = ((uint32_t(reinterpret_cast<uintptr_t>(sh)) + x0) >> 4) & 7;
            const bool edge = pre != 0 && (lane < 8 - pre || lane >= 64 - pre);
            auto put = [&](uint32_t at, u32x4 v, bool shared) {
                if (at + 16 <= data_end) {
                    if (shared) st16(sh + at, v);
                    else st_stream(sh, at, v);
                } else if (at < data_end) {
                    const gptr<uint8_t> d = as_global(sh);
                    for (uint32_t i = 0; i < data_end - at; ++i) d[at + i] = byte_of(v, int(i));
                }
            };
            if (X < rend) put(X, c0[r], edge);
            if (t0 + TB >= Sb && mr > 0 && threadIdx.x == BS - 1 && X + 16 < rend) put(X + 16, c1, true);
        }
        p ^= mr ? funnel16(c0[r], c1, mr) : c0[r];
        u32x4 qw;
        if (s > 0) qw = funnel16(c0[r], c1, uint32_t(s));
        else if (s == 0) qw = c0[r];
        else if (r <= 8 || s >= -16) qw = funnel16(cm, c0[r], uint32_t(s + 16));
        else qw = funnel16(from_prev_lane_or(cm, e2[r >= 8 ? r - 8 : 0]), cm, uint32_t(s + 32));
        q ^= star.d[r] < 0 ? qw : drop_word(qw, int64_t(star.d[r]) - w0);
    }
    *reinterpret_cast<u32x4*>(tp + 16 * threadIdx.x) = p;
    *reinterpret_cast<u32x4*>(tq + 16 * threadIdx.x) = q;
    __syncthreads();
    if (ND > 1 && t0 == 0) {
        if (wraps) {
            uint16_t v = 0;
#pragma unroll
            for (int r = 0; r < ND; ++r) v ^= star.d[r] == int32_t(threadIdx.x) ? uint16_t(0) : wq[r];
            *reinterpret_cast<uint16_t*>(tq + 2 * threadIdx.x) = v;
        }
        __syncthreads();
    }
    tile_store<true, BS>(sh + data_end + t0, tp, nbytes);
    tile_store<true, BS>(sh + data_end + Sb + t0, tq, nbytes);
}

// ----------------------------------------------------------------- recovery
// Row t (t >= 0) rebuilt as P ^ the other data rows, written back into the
// shards, and the stream written to K and V.  A block owns one tile of every
// row.  A surviving row's aligned chunks lie in one piece of K or V, so they
// go there straight from the registers they were loaded into; its at most 15
// bytes before the first and after the last whole chunk go byte by byte from
// block 0.  The rebuilt row is formed at the row's own alignment and goes
// through LDS.  Row t itself is never read.
template <int ND, int BS, bool FLAT>
__global__ __launch_bounds__(BS) void gs_recover_kv_kernel(uint8_t* sh, uint32_t Sb, uint32_t in_bytes, int t,
                                                           KvStream dst) {
    constexpr uint32_t TB = 16 * BS;
    __shared__ __attribute__((aligned(16))) uint8_t tile[TB + 16];
    const uint32_t t0 = blockIdx.x * TB;
    const uint32_t nbytes = Sb - t0 < TB ? Sb - t0 : TB;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t out_len = 2 * dst.kb;
    const __amdgpu_buffer_rsrc_t rs = chunk_rsrc(sh, (in_bytes + 15) & ~15u);
    // batch row i: data row i, or i + 1 from row t on (then P last)
    auto row_of = [&](int i) { return i + (t >= 0 && i >= t ? 1 : 0); };
    auto row_a = [&](int i) { return uint32_t(row_of(i)) * Sb + t0; };
    const bool live = 16 * threadIdx.x < nbytes + 16;
    u32x4 lo[ND], e1[ND];
#pragma unroll
    for (int i = 0; i < ND; ++i) {
        const uint32_t A = row_a(i), m = A & 15, my = A - m + 16 * threadIdx.x;
        lo[i] = chunk_load(rs, live ? my : kNoLoad);
        e1[i] = chunk_load(rs, live && lane == 63 && m ? my + 16 : kNoLoad);
    }
    __builtin_amdgcn_sched_barrier(0);
    u32x4 acc = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < ND; ++i) {
        const uint32_t A = row_a(i), m = A & 15, X = A - m + 16 * threadIdx.x;
        acc ^= m ? funnel16(lo[i], from_next_lane_or(lo[i], e1[i]), m) : lo[i];
        const uint32_t r0 = A - t0;
        if (row_of(i) < ND && X >= r0 && X + 16 <= r0 + Sb && X + 16 <= out_len)
            kv_put<FLAT>(dst, X, lo[i]);
    }
    if (blockIdx.x == 0) {
        for (uint32_t u = threadIdx.x; u < 32 * ND; u += BS) {
            const uint32_t j = uint32_t(row_of(int(u >> 5)));
            if (j < uint32_t(ND)) kv_put_row_end<FLAT>(dst, sh, Sb, j, u & 31);
        }
    }
    if (t < 0) return;
    *reinterpret_cast<u32x4*>(tile + 16 * threadIdx.x) = acc;
    __syncthreads();
    tile_store<false, BS>(sh + uint32_t(t) * Sb + t0, tile, nbytes);
    kv_put_tile<FLAT, BS>(dst, tile, uint32_t(t) * Sb + t0, nbytes);
}

// ------------------------------------------------------------ pack and unpack
// The stream to rows (zeros past V) and back, for codes whose kernels work on
// the rows: one pass in place of the permuted copies and the pack (33 MB of
// stream: 9 us to the rows against 32, 7 us back against 31).  Four chunks a
// thread, a wave's 4 KiB in a row.
constexpr int kPackBS = 256, kPackN = 4;

template <bool FLAT, bool PACK>
__global__ __launch_bounds__(kPackBS) void kv_rows_kernel(KvStream s, uint8_t* rows, uint32_t nbytes) {
    const uint32_t x0 = blockIdx.x * (16 * kPackBS * kPackN) +
                        uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6))) * (1024 * kPackN);
    const uint32_t lane16 = 16 * (threadIdx.x & 63);
    if (x0 >= nbytes) return;
    u32x4 v[kPackN];
    if constexpr (PACK) {
        const KvReader<FLAT> in(s);
        const auto f = in.from(x0, x0 + 1024 * kPackN);
#pragma unroll
        for (int n = 0; n < kPackN; ++n) v[n] = in.load(x0 + n * 1024 + lane16, true, f);
#pragma unroll
        for (int n = 0; n < kPackN; ++n)
            if (x0 + n * 1024 + lane16 < nbytes) st_stream(rows, x0 + n * 1024 + lane16, v[n]);
    } else {
#pragma unroll
        for (int n = 0; n < kPackN; ++n) {
            const uint32_t x = x0 + n * 1024 + lane16;
            v[n] = ld_stream(rows, x < nbytes ? x : x0);
        }
#pragma unroll
        for (int n = 0; n < kPackN; ++n) {
            const uint32_t x = x0 + n * 1024 + lane16;
            if (x < nbytes) kv_put<FLAT>(s, x, v[n]);
        }
    }
}

// ---------------------------------------------------------------- host side
// Threads per tile: 512 (8 KiB tiles) up to eight rows and 256 past them, whose
// registers leave room for 12 waves a CU (16 rows of 8.2 MB, P and Q: 28.9 us
// against 30.9 with 128 threads and 38.8 with 512; ten rows of K and V, 134 MB:
// 65.5 against 68.3 and 74.7); 128 where those tiles would leave compute units
// idle (16 rows of 0.4 MB: 6.7 against 7.3 us with 256).
constexpr int wide_bs(int nd) { return nd > 8 ? 256 : 512; }
constexpr int kKvSmallBS = 128;
static bool small_tiles(int nd, uint64_t Sb) { return Sb < (nd > 8 ? 1u << 20 : 4u << 20); }

constexpr int kKvMaxRows = 12;   // backup from K and V (SGPRs spill from 15 rows on)

typedef void (*BackupKvFn)(KvStream, uint8_t*, uint32_t, GsStar);
typedef void (*RecoverKvFn)(uint8_t*, uint32_t, uint32_t, int, KvStream);

template <bool SMALL, PqSource SRC, int ND = SRC == kRows ? 9 : 1>
static BackupKvFn backup_kv_fn(int nd) {
    if constexpr (ND > (SRC == kRows ? kGsMaxRows : kKvMaxRows)) {
        return nullptr;
    } else {
        if (nd == ND) return &gs_backup_kv_kernel<ND, SMALL ? kKvSmallBS : wide_bs(ND), SRC>;
        return backup_kv_fn<SMALL, SRC, ND + 1>(nd);
    }
}
template <bool SMALL, bool FLAT, int ND = 1>
static RecoverKvFn recover_kv_fn(int nd) {
    if constexpr (ND > kGsMaxRows) {
        return nullptr;
    } else {
        if (nd == ND) return &gs_recover_kv_kernel<ND, SMALL ? kKvSmallBS : wide_bs(ND), FLAT>;
        return recover_kv_fn<SMALL, FLAT, ND + 1>(nd);
    }
}

// P and Q (and, from K and V, the data rows) of rows of Sb bytes.
template <PqSource SRC>
static int launch_pq(const KvStream& s, uint8_t* sh, int nd, int64_t S, int star_base, hipStream_t st, const char* fn) {
    const uint64_t Sb = uint64_t(S) * 2;
    const bool small = small_tiles(nd, Sb);
    const BackupKvFn f = small ? backup_kv_fn<true, SRC>(nd) : backup_kv_fn<false, SRC>(nd);
    const int bs = small ? kKvSmallBS : wide_bs(nd);
    hipLaunchKernelGGL(f, dim3(blocks_for(int64_t(Sb), 16 * bs)), dim3(bs), 0, st, s, sh, uint32_t(Sb),
                       make_gs_star(star_base, S));
    return check_launch(fn);
}

int gs_rdp_parity_wide(uint16_t* sh, int nd, int64_t S, int star_base, hipStream_t st, const char* what) {
    return launch_pq<kRows>(KvStream{}, (uint8_t*)sh, nd, S, star_base, st, what);
}

// Whether the K/V kernels take this stripe: 1..max_nd data rows of at least 64
// words holding all of K and V, in a 16-byte-aligned tensor below 2 GiB.
static bool kv_rows_ok(const KvStream& s, const void* shards, int nd, int max_nd, int64_t S) {
    if (nd < 1 || nd > max_nd || S < 64 || !aligned16(shards)) return false;
    const uint64_t Sb = uint64_t(S) * 2;
    return uint64_t(nd + 2) * Sb <= (uint64_t(1) << 31) - 16 && 2 * uint64_t(s.kb) <= uint64_t(nd) * Sb;
}

static KvDims gs_dims(const kvec_kv_bhtd* kv) {
    return KvDims{kv->B, kv->H, kv->T, kv->head_bytes, kv->stride_b, kv->stride_h, kv->stride_t};
}

}  // namespace kvec

using namespace kvec;

extern "C" int kvec_gs_rdp_backup_kv(const kvec_kv_bhtd* kv, void* shards, int nd, int S, int star_base,
                                     void* stream) {
    static const char* fn = "kvec_gs_rdp_backup_kv";
    if (!kv || !shards) return set_error(KVEC_EINVAL, "%s: null pointer", fn);
    KvStream s{};
    bool flat = false;
    if (!make_kv_stream(&s, &flat, kv->k, kv->v, gs_dims(kv)) || !kv_rows_ok(s, shards, nd, kKvMaxRows, S))
        return set_error(KVEC_EUNSUPPORTED, "%s: layout or stripe not built", fn);
    if (!kv->k || !kv->v) return set_error(KVEC_EINVAL, "%s: null K or V", fn);
    const uint64_t Sb = uint64_t(S) * 2;
    const Span w = {shards, uint64_t(nd + 2) * Sb, "shards", -1};
    const Span r[2] = {{kv->k, s.ext, "k", -1}, {kv->v, s.ext, "v", -1}};
    if (int rc = check_no_alias(&w, 1, r, 2, fn)) return rc;
    const hipStream_t st = as_stream(stream);
    return flat ? launch_pq<kFlat>(s, (uint8_t*)shards, nd, S, star_base, st, fn)
                : launch_pq<kTokens>(s, (uint8_t*)shards, nd, S, star_base, st, fn);
}

extern "C" int kvec_gs_rdp_recover_kv(void* shards, const kvec_kv_bhtd* kv, int nd, int S, int star_base, int missing_a,
                                      int missing_b, void* stream) {
    static const char* fn = "kvec_gs_rdp_recover_kv";
    if (!kv || !shards) return set_error(KVEC_EINVAL, "%s: null pointer", fn);
    KvStream s{};
    bool flat = false;
    if (!make_kv_stream(&s, &flat, kv->k, kv->v, gs_dims(kv)) || !kv_rows_ok(s, shards, nd, kGsMaxRows, S))
        return set_error(KVEC_EUNSUPPORTED, "%s: layout or stripe not built", fn);
    if (!kv->k || !kv->v) return set_error(KVEC_EINVAL, "%s: null K or V", fn);
    const uint64_t Sb = uint64_t(S) * 2;
    int t = -1;
    if (int rc = gs_recover_row(nd, S, star_base, missing_a, missing_b, fn, &t)) return rc;
    const Span w[3] = {{shards, uint64_t(nd + 2) * Sb, "shards", -1}, {kv->k, s.ext, "k", -1}, {kv->v, s.ext, "v", -1}};
    if (int rc = check_no_alias(w, 3, nullptr, 0, fn)) return rc;
    const bool small = small_tiles(nd, Sb);
    const RecoverKvFn f = small ? (flat ? recover_kv_fn<true, true>(nd) : recover_kv_fn<true, false>(nd))
                                : (flat ? recover_kv_fn<false, true>(nd) : recover_kv_fn<false, false>(nd));
    const int bs = small ? kKvSmallBS : wide_bs(nd);
    hipLaunchKernelGGL(f, dim3(blocks_for(int64_t(Sb), 16 * bs)), dim3(bs), 0, as_stream(stream), (uint8_t*)shards,
                       uint32_t(Sb), uint32_t(uint64_t(nd + 1) * Sb), t, s);
    return check_launch(fn);
}

template <bool PACK>
static int kv_rows(const kvec_kv_bhtd* kv, void* rows, int64_t nbytes, void* stream, const char* fn) {
    if (!kv || !rows) return set_error(KVEC_EINVAL, "%s: null pointer", fn);
    KvStream s{};
    bool flat = false;
    if (!make_kv_stream(&s, &flat, kv->k, kv->v, gs_dims(kv)) || !aligned16(rows) || nbytes % 16 ||
        nbytes < 2 * int64_t(s.kb) || nbytes >= (int64_t(1) << 31))
        return set_error(KVEC_EUNSUPPORTED, "%s: layout not built", fn);
    if (!kv->k || !kv->v) return set_error(KVEC_EINVAL, "%s: null K or V", fn);
    const Span a[3] = {{rows, uint64_t(nbytes), "rows", -1}, {kv->k, s.ext, "k", -1}, {kv->v, s.ext, "v", -1}};
    if (int rc = PACK ? check_no_alias(a, 1, a + 1, 2, fn) : check_no_alias(a, 3, nullptr, 0, fn)) return rc;
    const uint32_t n = PACK ? uint32_t(nbytes) : 2 * s.kb;
    auto kern = flat ? &kv_rows_kernel<true, PACK> : &kv_rows_kernel<false, PACK>;
    hipLaunchKernelGGL(kern, dim3(blocks_for(n, 16 * kPackBS * kPackN)), dim3(kPackBS), 0, as_stream(stream), s,
                       (uint8_t*)rows, n);
    return check_launch(fn);
}

extern "C" int kvec_kv_pack_bhtd(const kvec_kv_bhtd* kv, void* rows, int64_t rows_bytes, void* stream) {
    return kv_rows<true>(kv, rows, rows_bytes, stream, "kvec_kv_pack_bhtd");
}

extern "C" int kvec_kv_unpack_bhtd(const void* rows, int64_t rows_bytes, const kvec_kv_bhtd* kv, void* stream) {
    return kv_rows<false>(kv, const_cast<void*>(rows), rows_bytes, stream, "kvec_kv_unpack_bhtd");
}
