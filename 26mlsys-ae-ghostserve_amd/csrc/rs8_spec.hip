// rs8_spec.hip -- systematic Reed-Solomon over GF(2^8) (poly 0x11D) with the
// Cauchy parity block C[i][j] = 1 / ((k+i) ^ j), i < m, j < k.
//
// Encode and decode are the same operation: out_o = XOR_j M[o][j] * in_j over
// separate shard buffers, with M = C for encode and, for decode, the rows of
// the inverse of the surviving k x k block of [I; C] (and C times it for an
// erased parity shard), computed on the host.
//
// The constant multiply is the v_perm_b32 split-table product of gf8.h.  Per 4
// data bytes: 5 ops to extract the fields (shared by all outputs) and 3 v_perm
// + 3 XOR per coefficient, with the tables held in registers -- no LDS or
// memory lookups.
#include "gf8.h"
#include "kv_stream.h"

namespace kvec {

// The coefficient tables are staged in LDS and read at their point of use:
// held in SGPRs from the kernel arguments, 6*k*m dwords next to the shard
// buffer resources overflow the SGPR file and get spilled (and kernels that
// spilled SGPRs have given run-to-run different results).
template <int NIN, int NOUT, int V>
__global__ __launch_bounds__(kRs8BS) void gf8_mix_kernel(Ptrs<kRs8MaxK> in, Ptrs<kRs8MaxM> out,
                                                         Gf8Mix mix, uint32_t S, uint32_t nvec) {
    __shared__ uint32_t lds_tab[NIN * NOUT][6];
    for (int i = threadIdx.x; i < NIN * NOUT * 6; i += kRs8BS) lds_tab[i / 6][i % 6] = mix.t[i / 6][i % 6];
    __syncthreads();
    auto tab = [&](int c) -> const uint32_t* { return lds_tab[c]; };
    const uint32_t u0 = blockIdx.x * (kRs8BS * V) + threadIdx.x;
    u32x4 acc[V][NOUT];
#pragma unroll
    for (int v = 0; v < V; ++v)
#pragma unroll
        for (int o = 0; o < NOUT; ++o) acc[v][o] = u32x4{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < NIN; ++j) {
        const ShardView<true> sv(in.p[j], S);
        u32x4 x[V];
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const uint32_t u = u0 + v * kRs8BS;
            x[v] = sv.load(0, (u < nvec ? u : 0u) << 4);
        }
#pragma unroll
        for (int v = 0; v < V; ++v) {
            Gf8Fields f[4];
            gf8_fields16(x[v], f);
#pragma unroll
            for (int o = 0; o < NOUT; ++o) acc[v][o] = gf8_fma16(acc[v][o], f, tab(o * NIN + j));
        }
    }
#pragma unroll
    for (int o = 0; o < NOUT; ++o) {
        const ShardView<true> so(out.p[o], S);
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const uint32_t u = u0 + v * kRs8BS;
            if (u < nvec) so.store(0, u << 4, acc[v][o]);
        }
    }
}

// ------------------------------------------------- any shape, and K and V
// NOUT outputs over any number of inputs, in a loop: a thread owns V 16-byte
// windows of every shard, two inputs' windows are in flight, and the loop is
// unrolled by two so that none is copied (an odd input count gets one with
// zero coefficients).  Tables as above, staged in LDS input by input.
//   kShards   separate shards; outputs in groups of NOUT by blockIdx.y
//   kEncode   rs.forward_encode_kv: the inputs are the rows of the stream
//             K || V || zeros, which the loads also write into the shard
//             tensor's data rows; the outputs are its parity rows
//   kDecode   rs.backwards_decode_kv: inputs and outputs are rows of the shard
//             tensor; the data rows among both also go to K and V
// The packed forms move each byte once, where pack, code and split moved K, V
// and the rows two to three times.  Rows are multiples of 16 bytes.  Bound by
// HBM (201 MB stream of separate shards, against one output at a time through
// L2): 5.3-5.9 TB/s; of K and V 5.0-5.3 TB/s, 59 us for the 313 MB of RS(6, 2).
enum Rs8Mode { kShards, kEncode, kDecode };

template <Rs8Mode MODE>
struct Rs8Io;
template <>
struct Rs8Io<kShards> {
    Ptrs<kRs8MaxK> in;
    Ptrs<kRs8MaxM> out;
};
template <>
struct Rs8Io<kEncode> {
    KvStream kv;
    uint8_t* sh;
    int k;
};
template <>
struct Rs8Io<kDecode> {
    KvStream kv;
    uint8_t* sh;
    int k;
    uint8_t in[kRs8MaxK], out[kRs8MaxM];   // rows
    uint32_t sh_bytes;
};

constexpr int kRs8LoopBS = 256;

template <int NOUT, int V, Rs8Mode MODE, bool NT = true>
__global__ __launch_bounds__(kRs8LoopBS) void gf8_loop_kernel(Rs8Io<MODE> io, Gf8Mix mix, int nin, int nout,
                                                              uint32_t S) {
    constexpr uint32_t TB = 16 * kRs8LoopBS * V, WB = 1024 * V;
    static_assert((TB & (TB - 1)) == 0, "columns of the last tile stay below 2^32");
    __shared__ __attribute__((aligned(16))) uint32_t tab[kRs8MaxK][NOUT][6];   // nin is even or padded
    const int o0 = int(blockIdx.y) * NOUT, nj = (nin + 1) & ~1;
    for (int e = threadIdx.x; e < nj * NOUT * 6; e += kRs8LoopBS) {
        const int j = e / (NOUT * 6), o = e / 6 % NOUT, d = e % 6;
        tab[j][o][d] = j < nin && o0 + o < nout ? mix.t[(o0 + o) * nin + j][d] : 0u;
    }
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t t0 = blockIdx.x * TB;
    const uint32_t wb = t0 + uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6))) * WB;
    // shards of up to 4 GiB: the tile divides 2^32, so a column never wraps
    auto col = [&](int v) { return wb + v * 1024 + 16 * lane; };
    __amdgpu_buffer_rsrc_t rs;
    if constexpr (MODE == kDecode) rs = chunk_rsrc(io.sh, io.sh_bytes);
    // the stream chunk at X to K or V
    auto to_kv = [&](uint32_t X, u32x4 v) {
        if constexpr (MODE == kDecode)
            if (X < 2 * io.kv.kb) st_stream(kv_at<true>(io.kv, X), 0, v);
    };
    auto load = [&](int j, u32x4 (&x)[V]) {
        if (j >= nin) return;   // uniform
        if constexpr (MODE == kShards) {
#pragma unroll
            for (int v = 0; v < V; ++v) {
                const uint8_t* p = io.in.p[j];
                const uint32_t c = col(v) < S ? col(v) : 0u;
                x[v] = NT ? ld_stream(p, c) : ld16(p + c);
            }
        } else if constexpr (MODE == kDecode) {
            const uint32_t r0 = uint32_t(io.in[j]) * S;
#pragma unroll
            for (int v = 0; v < V; ++v) x[v] = chunk_load(rs, r0 + col(v));
        } else {
            const uint32_t kb = io.kv.kb, X = uint32_t(j) * S + wb;
            const bool in_v = X >= kb;
            if (X + WB <= kb || (in_v && X + WB <= 2 * kb)) {   // uniform: one piece of K or of V
                const uint8_t* p = in_v ? io.kv.V + (X - kb) : io.kv.K + X;
#pragma unroll
                for (int v = 0; v < V; ++v) x[v] = ld_stream(p + v * 1024, 16 * lane);
            } else {
#pragma unroll
                for (int v = 0; v < V; ++v) {
                    const uint32_t y = X + v * 1024 + 16 * lane, c = y < 2 * kb - 16 ? y : 2 * kb - 16;
                    const u32x4 w = ld16(c >= kb ? io.kv.V + (c - kb) : io.kv.K + c);
                    const u32x4 zero = {0, 0, 0, 0};
                    x[v] = y < 2 * kb ? w : zero;
                }
            }
        }
    };
    u32x4 acc[V][NOUT];
#pragma unroll
    for (int v = 0; v < V; ++v)
#pragma unroll
        for (int o = 0; o < NOUT; ++o) acc[v][o] = u32x4{0, 0, 0, 0};
    auto use = [&](int j, const u32x4 (&x)[V]) {
        if constexpr (MODE == kEncode) {
#pragma unroll
            for (int v = 0; v < V; ++v)
                if (col(v) < S && j < nin) st_stream(io.sh + uint32_t(j) * S, col(v), x[v]);
        } else if constexpr (MODE == kDecode) {
            if (j < nin && io.in[j] < io.k) {   // uniform
#pragma unroll
                for (int v = 0; v < V; ++v)
                    if (col(v) < S) to_kv(uint32_t(io.in[j]) * S + col(v), x[v]);
            }
        }
#pragma unroll
        for (int v = 0; v < V; ++v) {
            Gf8Fields f[4];
            gf8_fields16(x[v], f);
#pragma unroll
            for (int o = 0; o < NOUT; ++o) acc[v][o] = gf8_fma16(acc[v][o], f, tab[j][o]);
        }
    };
    u32x4 xa[V], xb[V];
#pragma unroll
    for (int v = 0; v < V; ++v) xa[v] = xb[v] = u32x4{0, 0, 0, 0};
    load(0, xa);
    load(1, xb);
    __syncthreads();   // tab
    for (int j = 0; j < nin; j += 2) {
        use(j, xa);
        load(j + 2, xa);
        use(j + 1, xb);
        load(j + 3, xb);
    }
#pragma unroll
    for (int o = 0; o < NOUT; ++o) {
        if (o0 + o >= nout) break;   // uniform
#pragma unroll
        for (int v = 0; v < V; ++v) {
            if (col(v) >= S) continue;
            if constexpr (MODE == kShards) {
                st_stream(io.out.p[o0 + o], col(v), acc[v][o]);
            } else if constexpr (MODE == kEncode) {
                st_stream(io.sh + uint32_t(io.k + o) * S, col(v), acc[v][o]);
            } else {
                st_stream(io.sh + uint32_t(io.out[o]) * S, col(v), acc[v][o]);
                if (io.out[o] < io.k) to_kv(uint32_t(io.out[o]) * S + col(v), acc[v][o]);
            }
        }
    }
}

// One window per thread, but two where three or four outputs are decoded to K
// and V (10 rows, four lost, 67 MB: 42 against 50 us; 8 rows, three lost 33
// against 42).  Elsewhere one is faster: 134 MB of K and V in six rows, encode
// 59 against 61 us, two lost 62 against 69, one lost 58 against 62; RS(10, 4) of
// 67 MB 34 against 38.  128 and 512 threads: within 5 % either way.
template <Rs8Mode MODE, bool NT = true>
static int launch_loop(const Rs8Io<MODE>& io, const Gf8Mix& mix, int nin, int nout, uint32_t S, hipStream_t st,
                       const char* what) {
    constexpr int W = MODE == kDecode ? 2 : 1;
    auto go = [&](auto kern, int n, int v) {
        hipLaunchKernelGGL(kern, dim3(blocks_for(S, 16 * kRs8LoopBS * v), blocks_for(nout, n)), dim3(kRs8LoopBS), 0, st,
                           io, mix, nin, nout, S);
    };
    switch (nout) {
        case 1: go(&gf8_loop_kernel<1, 1, MODE, NT>, 1, 1); break;
        case 2: go(&gf8_loop_kernel<2, 1, MODE, NT>, 2, 1); break;
        case 3: go(&gf8_loop_kernel<3, W, MODE, NT>, 3, W); break;
        default: go(&gf8_loop_kernel<4, W, MODE, NT>, 4, W); break;
    }
    return check_launch(what);
}

// One output at a time, inputs re-read through L2: one input and one output (shards
// of 33 MB 11.0 us against 13.9 by the loop, which pairs inputs, 100 MB 33.4 against
// 35.8, 201 MB 67.0 against 69.5), and shards of 4 GiB and more, past the loop
// kernel's 32-bit columns (of 2 GiB, this against the loop: RS(8, 2) 5.2 against 3.4
// ms, (10, 4) 12.0 against 5.0).
__global__ __launch_bounds__(kRs8BS) void gf8_mix_generic_kernel(Ptrs<kRs8MaxK> in,
                                                                 Ptrs<kRs8MaxM> out, Gf8Mix mix,
                                                                 int nin, int nout, uint64_t nvec) {
    const uint64_t u = uint64_t(blockIdx.x) * kRs8BS + threadIdx.x;
    if (u >= nvec) return;
    for (int o = 0; o < nout; ++o) {
        u32x4 acc = {0, 0, 0, 0};
        for (int j = 0; j < nin; ++j) {
            const u32x4 x = ld16(in.p[j] + (u << 4));
            const uint32_t w[4] = {x.x, x.y, x.z, x.w};
            uint32_t r[4];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                r[q] = gf8_mul4(w[q] & 0x07070707u, (w[q] >> 3) & 0x07070707u,
                                (w[q] >> 6) & 0x03030303u, mix.t[o * nin + j]);
            acc ^= u32x4{r[0], r[1], r[2], r[3]};
        }
        st_stream(out.p[o], u << 4, acc);
    }
}

typedef void (*MixFn)(Ptrs<kRs8MaxK>, Ptrs<kRs8MaxM>, Gf8Mix, uint32_t, uint32_t);

// Large shards of some shapes keep the straight-line kernel: two outputs of four
// to six inputs from 60 MiB on (512 MiB stream: RS(4, 2) 127-129 against 136 us
// for the loop, (5, 2) 123 against 125, (6, 2) 115.5 against 118.4; 201 MB: (4, 2)
// 53 against 51 us, (6, 2) 47.0 against 46.5), two outputs of eight from 40 MiB
// (shards of 34 MB 57-59 against 56-57 us, 42 MB 69 against 71, 55 MB 88 against 93,
// 64 MiB 106 against 113-119, 201 MB 315 against 351, 805 MB 1293 against 1350), one
// of ten from 48 MiB (42 MB 78 against 76, 59 MB 105 against 108, 134 MB 242
// against 250).  On the other shapes that had one the loop is as fast or faster,
// 1 MB to 2 GiB shards: (4, 1), (5, 1), (6, 1), (8, 1) and (5, 3) within 2 % from 34
// MB on, (10, 2) of 20 MB 48 against 42 us and of 54 MB 115 against 111, (10, 4) of
// 54 MB 128 against 122.
struct MixKern {
    MixFn fn;
    int vec;   // 16-byte windows of a thread
};
static MixKern mix_kern(int nin, int nout, uint64_t S) {
    const MixKern none = {nullptr, 0};
    if (!fits_buffer(S) || S < (nin == 8 ? 40u << 20 : nin == 10 ? 48u << 20 : 60u << 20)) return none;
    if (nout == 1 && nin == 10) return {&gf8_mix_kernel<10, 1, 2>, 2};
    if (nout != 2) return none;
    switch (nin) {
        case 4: return {&gf8_mix_kernel<4, 2, 2>, 2};
        case 5: return {&gf8_mix_kernel<5, 2, 2>, 2};
        case 6: return {&gf8_mix_kernel<6, 2, 2>, 2};
        case 8: return {&gf8_mix_kernel<8, 2, 1>, 1};
        default: return none;
    }
}

// The loop's loads from separate shards: ordinary ones up to 128 MiB of inputs and
// outputs, which may still lie in the 256 MB memory-side cache from what wrote
// or read them, non-temporal ones past it (three sets in turn, ordinary against
// non-temporal: 2 shards to 1 of 17 MB 8.4 against 10.7 us, 3 to 2 of 11 MB 10.1
// against 12.0; 4 to 1 of 50 MB 45.7 against 42.6, 16 to 2 of 13 MB 43.5
// against 40.8).
constexpr uint64_t kRs8CachedBytes = 128u << 20;

static int launch_mix(uint8_t* const* in, int nin, uint8_t* const* out, int nout,
                      const uint8_t* M /* nout x nin */, int64_t S, hipStream_t st,
                      const char* what) {
    Ptrs<kRs8MaxK> pi{};
    Ptrs<kRs8MaxM> po{};
    Gf8Mix mix{};
    for (int j = 0; j < nin; ++j) pi.p[j] = in[j];
    for (int o = 0; o < nout; ++o) {
        po.p[o] = out[o];
        for (int j = 0; j < nin; ++j) perm_tables(M[o * nin + j], mix.t[o * nin + j]);
    }
    if (S == 0 || nout == 0) return KVEC_OK;
    if (const MixKern kern = mix_kern(nin, nout, uint64_t(S)); kern.fn) {
        const uint32_t nvec = uint32_t(S / 16);
        hipLaunchKernelGGL(kern.fn, dim3(blocks_for(nvec, kRs8BS * kern.vec)), dim3(kRs8BS), 0, st, pi, po, mix,
                           uint32_t(S), nvec);
    } else if (fits_buffer(uint64_t(S)) && nin * nout > 1) {   // 32-bit columns
        const Rs8Io<kShards> io = {pi, po};
        return uint64_t(nin + nout) * uint64_t(S) <= kRs8CachedBytes
                       ? launch_loop<kShards, false>(io, mix, nin, nout, uint32_t(S), st, what)
                       : launch_loop<kShards, true>(io, mix, nin, nout, uint32_t(S), st, what);
    } else {
        const uint64_t nvec = uint64_t(S) / 16;
        hipLaunchKernelGGL(gf8_mix_generic_kernel, dim3(unsigned((nvec + kRs8BS - 1) / kRs8BS)),
                           dim3(kRs8BS), 0, st, pi, po, mix, nin, nout, nvec);
    }
    return check_launch(what);
}

static int check_rs8(int k, int m, int64_t S, const char* fn) {
    if (k < 1 || m < 0 || k > kRs8MaxK || m > kRs8MaxM || k * m > kRs8MaxCoef)
        return set_error(KVEC_EINVAL, "%s: k=%d m=%d (k <= %d, m <= %d, k*m <= %d)", fn, k, m, kRs8MaxK,
                         kRs8MaxM, kRs8MaxCoef);
    if (S < 0 || S % 16) return set_error(KVEC_EINVAL, "%s: shard_bytes=%lld must be a multiple of 16", fn,
                                          (long long)S);
    return KVEC_OK;
}

}  // namespace kvec

using namespace kvec;

extern "C" int kvec_rs8_cauchy(int k, int m, uint8_t* C) {
    if (k < 1 || m < 0 || k + m > 256 || !C) return set_error(KVEC_EINVAL, "kvec_rs8_cauchy: k=%d m=%d", k, m);
    cauchy(k, m, C);
    return KVEC_OK;
}

extern "C" int kvec_rs8_encode(const void* const* data, int k, void* const* parity, int m,
                               int64_t shard_bytes, void* stream) {
    int rc = check_rs8(k, m, shard_bytes, "kvec_rs8_encode");
    if (rc) return rc;
    if (m == 0) return KVEC_OK;
    if (!data || !parity) return set_error(KVEC_EINVAL, "kvec_rs8_encode: null pointer array");
    uint8_t* in[kRs8MaxK];
    uint8_t* out[kRs8MaxM];
    for (int j = 0; j < k; ++j) {
        if (!data[j] || !aligned16(data[j]))
            return set_error(KVEC_EINVAL, "kvec_rs8_encode: data[%d] null or not 16-byte aligned", j);
        in[j] = (uint8_t*)data[j];
    }
    for (int i = 0; i < m; ++i) {
        if (!parity[i] || !aligned16(parity[i]))
            return set_error(KVEC_EINVAL, "kvec_rs8_encode: parity[%d] null or not 16-byte aligned", i);
        out[i] = (uint8_t*)parity[i];
    }
    {
        Span w[kRs8MaxM], r[kRs8MaxK];
        for (int i = 0; i < m; ++i) w[i] = Span{out[i], uint64_t(shard_bytes), "parity", i};
        for (int j = 0; j < k; ++j) r[j] = Span{in[j], uint64_t(shard_bytes), "data", j};
        if ((rc = check_no_alias(w, m, r, k, "kvec_rs8_encode"))) return rc;
    }
    uint8_t C[kRs8MaxM * kRs8MaxK];
    cauchy(k, m, C);
    return launch_mix(in, k, out, m, C, shard_bytes, as_stream(stream), "kvec_rs8_encode");
}

extern "C" int kvec_rs8_decode(void* const* shards, int k, int m, int64_t shard_bytes,
                               const int32_t* erased, int n_erased, void* stream) {
    int rc = check_rs8(k, m, shard_bytes, "kvec_rs8_decode");
    if (rc) return rc;
    if (!shards || (n_erased > 0 && !erased))
        return set_error(KVEC_EINVAL, "kvec_rs8_decode: null pointer");
    bool er[kRs8MaxK + kRs8MaxM] = {};
    for (int q = 0; q < n_erased; ++q) {
        if (erased[q] < 0 || erased[q] >= k + m)
            return set_error(KVEC_EINVAL, "kvec_rs8_decode: erased index %d not in [0, %d)", erased[q], k + m);
        er[erased[q]] = true;
    }
    int ne = 0;
    for (int s = 0; s < k + m; ++s) {
        if (!shards[s] || !aligned16(shards[s]))
            return set_error(KVEC_EINVAL, "kvec_rs8_decode: shard %d null or not 16-byte aligned", s);
        ne += er[s];
    }
    if (ne == 0) return KVEC_OK;
    if (ne > m) return set_error(KVEC_EDECODE, "kvec_rs8_decode: %d erasures > m=%d", ne, m);
    {
        // the rebuilt shards must not share a byte with any other shard
        Span w[kRs8MaxM], r[kRs8MaxK + kRs8MaxM];
        int nw = 0, nr = 0;
        for (int s = 0; s < k + m; ++s)
            (er[s] ? w[nw++] : r[nr++]) = Span{shards[s], uint64_t(shard_bytes), "shard", s};
        if ((rc = check_no_alias(w, nw, r, nr, "kvec_rs8_decode"))) return rc;
    }
    int surv[kRs8MaxK], outs[kRs8MaxM], no = 0;
    uint8_t M[kRs8MaxM * kRs8MaxK];
    if (!rs8_decode_rows(k, m, er, surv, outs, &no, M))
        return set_error(KVEC_EDECODE, "kvec_rs8_decode: singular survivor block");
    uint8_t* in[kRs8MaxK];
    uint8_t* out[kRs8MaxM];
    for (int o = 0; o < no; ++o) out[o] = (uint8_t*)shards[outs[o]];
    for (int q = 0; q < k; ++q) in[q] = (uint8_t*)shards[surv[q]];
    return launch_mix(in, k, out, no, M, shard_bytes, as_stream(stream), "kvec_rs8_decode");
}

// The packed rows and the stream of rs.forward_encode_kv / backwards_decode_kv
// with these codes, or EUNSUPPORTED.  The encode only reads K and V, which may
// then be the same memory.
static int rs8_kv_stream(KvStream* s, const void* K, const void* V, int64_t half, const void* shards, int k, int m,
                         int64_t S, bool encode, const char* fn) {
    bool flat = false;
    if (m < 1 || S < 16 || !aligned16(shards) || half < 16 || uint64_t(k + m) * uint64_t(S) >= (uint64_t(1) << 31) ||
        S >= (int64_t(1) << 31) || !make_kv_stream(s, &flat, K, V, KvDims{1, 1, 1, half, 0, 0, 0}) ||
        2 * uint64_t(s->kb) > uint64_t(k) * uint64_t(S))
        return set_error(KVEC_EUNSUPPORTED, "%s: layout or stripe not built", fn);
    if (!K || !V) return set_error(KVEC_EINVAL, "%s: null K or V", fn);
    const Span w[3] = {{shards, uint64_t(k + m) * uint64_t(S), "shards", -1}, {K, s->kb, "K", -1}, {V, s->kb, "V", -1}};
    return encode ? check_no_alias(w, 1, w + 1, 2, fn) : check_no_alias(w, 3, nullptr, 0, fn);
}

extern "C" int kvec_rs8_encode_kv(const void* key_input, const void* value_input, int64_t kv_half_bytes, void* shards,
                                  int data_shards, int parity_shards, int64_t row_bytes, void* stream) {
    static const char* fn = "kvec_rs8_encode_kv";
    const int k = data_shards, m = parity_shards;
    int rc = check_rs8(k, m, row_bytes, fn);
    if (rc) return rc;
    if (!shards) return set_error(KVEC_EINVAL, "%s: null pointer", fn);
    Rs8Io<kEncode> io{};
    if (m > 4) return set_error(KVEC_EUNSUPPORTED, "%s: %d parity rows", fn, m);
    if ((rc = rs8_kv_stream(&io.kv, key_input, value_input, kv_half_bytes, shards, k, m, row_bytes, true, fn))) return rc;
    io.sh = (uint8_t*)shards;
    io.k = k;
    uint8_t C[kRs8MaxM * kRs8MaxK];
    cauchy(k, m, C);
    Gf8Mix mix{};
    for (int t = 0; t < k * m; ++t) perm_tables(C[t], mix.t[t]);
    return launch_loop<kEncode>(io, mix, k, m, uint32_t(row_bytes), as_stream(stream), fn);
}

extern "C" int kvec_rs8_recover_kv(void* shards, void* key_output, void* value_output, int64_t kv_half_bytes,
                                   int data_shards, int parity_shards, int64_t row_bytes, const int32_t* erased,
                                   int n_erased, void* stream) {
    static const char* fn = "kvec_rs8_recover_kv";
    const int k = data_shards, m = parity_shards;
    int rc = check_rs8(k, m, row_bytes, fn);
    if (rc) return rc;
    if (!shards || (n_erased > 0 && !erased)) return set_error(KVEC_EINVAL, "%s: null pointer", fn);
    bool er[kRs8MaxK + kRs8MaxM] = {};
    int ne = 0;
    for (int q = 0; q < n_erased; ++q) {
        if (erased[q] < 0 || erased[q] >= k + m)
            return set_error(KVEC_EINVAL, "%s: erased index %d not in [0, %d)", fn, erased[q], k + m);
        ne += !er[erased[q]];
        er[erased[q]] = true;
    }
    if (ne > m) return set_error(KVEC_EDECODE, "%s: %d erasures > m=%d", fn, ne, m);
    Rs8Io<kDecode> io{};
    if (ne < 1 || ne > 4) return set_error(KVEC_EUNSUPPORTED, "%s: %d erasures", fn, ne);
    if ((rc = rs8_kv_stream(&io.kv, key_output, value_output, kv_half_bytes, shards, k, m, row_bytes, false, fn))) return rc;
    int surv[kRs8MaxK], outs[kRs8MaxM], no = 0;
    uint8_t M[kRs8MaxM * kRs8MaxK];
    if (!rs8_decode_rows(k, m, er, surv, outs, &no, M))
        return set_error(KVEC_EDECODE, "%s: singular survivor block", fn);
    io.sh = (uint8_t*)shards;
    io.sh_bytes = uint32_t(uint64_t(k + m) * uint64_t(row_bytes));
    io.k = k;
    for (int j = 0; j < k; ++j) io.in[j] = uint8_t(surv[j]);
    for (int o = 0; o < no; ++o) io.out[o] = uint8_t(outs[o]);
    Gf8Mix mix{};
    for (int t = 0; t < no * k; ++t) perm_tables(M[t], mix.t[t]);
    return launch_loop<kDecode>(io, mix, k, no, uint32_t(row_bytes), as_stream(stream), fn);
}
