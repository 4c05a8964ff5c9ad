"""The reference's star-diagonal "RDP" code, signature-compatible with
benchmark/rdp/main.py.

``rdp_kernel`` stands in for the pybind module ``rdp_kernel_rdp_parallel``
(benchmark/rdp/kernel.cu:525-538).  The P/Q bytes are those of the reference.
Its two-row "recovery" is reproduced as the reference observably behaves: the
lower row is rebuilt from P and the other row keeps its input bytes (the
reference's ring walk is overwritten by its final rebuild-from-P kernels), so
it recovers nothing when two data rows are really lost.

``scheme="spec"`` keeps the same functions, arguments and returned dicts but
codes the shard tensor with textbook RDP (Corbett et al., FAST 2004) over the
smallest prime p > num_data_shards (p = 7 for six data shards): the data rows
are shards, row nd is P and row nd+1 is Q, and fused_recovery_full_kv then
rebuilds any two lost rows (data, P or Q) byte-exact.  Its shard size is the
reference's rounded up so that every shard row splits into p-1 RDP rows of a
whole number of 16-byte cells.

K/V may be any 2-byte dtype (coded as raw bits; results come back in the input
dtype).
"""
from __future__ import annotations

import torch

from . import _lib, spec


def _stream(t: torch.Tensor) -> int:
    return _lib.stream_handle(t.device)


class _RdpKernel:
    """The reference module ``rdp_kernel_rdp_parallel``."""

    @staticmethod
    def fused_backup_full_kv(K_TN, V_TN, shards, num_data_shards, shard_size, T, n, star_base):
        _lib.require_cuda(K_TN, V_TN, shards, what="fused_backup_full_kv tensor")
        _lib.call("kvec_gs_rdp_backup", K_TN.data_ptr(), V_TN.data_ptr(), shards.data_ptr(),
                  int(num_data_shards), int(shard_size), int(T), int(n), int(star_base),
                  _stream(shards))

    @staticmethod
    def fused_recovery_full_kv(shards, out_half_TN, num_data_shards, shard_size, T, n, star_base,
                               missing_a, missing_b):
        _lib.require_cuda(shards, out_half_TN, what="fused_recovery_full_kv tensor")
        _lib.call("kvec_gs_rdp_recover", shards.data_ptr(), out_half_TN.data_ptr(),
                  int(num_data_shards), int(shard_size), int(T), int(n), int(star_base),
                  int(missing_a), int(missing_b), _stream(shards))


rdp_kernel = _RdpKernel()


def determine_shard_size_words(total_words: int, num_data_shards: int):
    """benchmark/rdp/main.py:21-27."""
    if num_data_shards <= 0:
        raise ValueError("num_data_shards must be > 0")
    pad = (num_data_shards - (total_words % num_data_shards)) % num_data_shards
    padded_total = total_words + pad
    shard_size = padded_total // num_data_shards
    return shard_size, pad


SCHEMES = ("ghostserve", "spec")


def spec_prime(num_data_shards: int) -> int:
    """Smallest odd prime p with p - 1 >= num_data_shards."""
    p = max(3, int(num_data_shards) + 1)
    while any(p % q == 0 for q in range(2, int(p ** 0.5) + 1)):
        p += 1
    return p


def spec_shard_size_words(total_words: int, num_data_shards: int, p: int):
    """The reference's shard size rounded up so that a shard row splits into
    p-1 RDP rows of a multiple of 16 bytes (8 words) each.  Returns
    (shard_size, pad_words)."""
    S, _ = determine_shard_size_words(total_words, num_data_shards)
    q = 8 * (p - 1)
    S = -(-S // q) * q
    return S, num_data_shards * S - total_words


def _rows_u8(shards: torch.Tensor):
    """The rows of a [(rows), S] uint16 shard tensor as byte tensors."""
    b = shards.view(torch.uint8).view(shards.shape[0], -1)
    return [b[i] for i in range(shards.shape[0])]


def _check_scheme(scheme: str):
    if scheme not in SCHEMES:
        raise ValueError(f"scheme must be one of {SCHEMES}, not {scheme!r}")


def _token_major(keys, values):
    """[T, B*H*D] copies of K and V indexed [B, H, T, D]."""
    return tuple(x.permute(2, 0, 1, 3).contiguous().view(x.shape[2], -1) for x in (keys, values))


def _copies_are_faster(B: int, H: int, T: int, head_bytes: int) -> bool:
    """Large K and V [B, H, T, head] of many heads of 16 bytes: each chunk that a
    wave of the one-pass kernels moves is in another head's plane (backup of six
    rows, K of 67 MB, copies against one pass: 128 heads 268 against 192 us, 256
    heads 186 against 241, 1024 heads 172 against 217; 256 heads of 12 MB 63
    against 55, 17 MB 75 against 77)."""
    return head_bytes == 16 and B * H >= 192 and B * H * T * 16 >= 14_000_000


def fused_backup_full_kv(keys_bhtd: torch.Tensor, values_bhtd: torch.Tensor,
                         num_data_shards: int, star_base: int = 0, scheme: str = "ghostserve"):
    """benchmark/rdp/main.py:44-92: token-major pack + P/Q in one call.
    scheme="spec": textbook RDP P/Q instead of the star-diagonal code."""
    _check_scheme(scheme)
    if not (keys_bhtd.is_cuda and values_bhtd.is_cuda):
        raise ValueError("keys/values must be CUDA tensors.")
    if keys_bhtd.dtype != values_bhtd.dtype or keys_bhtd.element_size() != 2:
        raise ValueError("keys/values must be fp16 (or another 2-byte dtype).")
    if keys_bhtd.shape != values_bhtd.shape:
        raise ValueError("K and V shapes must match [B,H,T,D].")
    if num_data_shards <= 0:
        raise ValueError("num_data_shards must be > 0")

    B, H, T, D = keys_bhtd.shape
    n = B * H * D
    total_words = 2 * T * n

    nd = int(num_data_shards)
    p = spec_prime(nd) if scheme == "spec" else 0
    if scheme == "spec":
        shard_size, pad_words = spec_shard_size_words(total_words, nd, p)
    else:
        shard_size, pad_words = determine_shard_size_words(total_words, nd)
    # one pass over K and V where they lie, when the layout allows it (what can
    # be known here: up to twelve rows of 64 words and more) and unless copies
    # are faster (never when a token's heads are adjacent); else token-major
    # copies, then the pack and the code
    kv = None
    if (scheme == "spec" or (nd <= 12 and shard_size >= 64)) and not (
            _copies_are_faster(B, H, T, D * 2) and keys_bhtd.stride(1 if H > 1 else 0) != D):
        kv = _lib.kv_bhtd(keys_bhtd, values_bhtd)
    # (the copies first, so that the host prepares the rest behind them)
    copies = _token_major(keys_bhtd, values_bhtd) if kv is None else None
    shards = torch.empty((nd + 2, shard_size), dtype=torch.uint16, device=keys_bhtd.device)
    t0 = torch.cuda.Event(enable_timing=True)
    t1 = torch.cuda.Event(enable_timing=True)
    direct = False
    if kv is not None:
        t0.record()
        if scheme == "spec":
            direct = _lib.call_if_built("kvec_kv_pack_bhtd", kv, shards.data_ptr(),
                                        2 * nd * int(shard_size), _stream(shards))
        else:
            direct = _lib.call_if_built("kvec_gs_rdp_backup_kv", kv, shards.data_ptr(), nd,
                                        int(shard_size), int(star_base), _stream(shards))
    if not direct:
        K_TN, V_TN = copies or _token_major(keys_bhtd, values_bhtd)
        # the reference zero-fills everything; only the padding words are read
        # before being written
        shards.view(-1).view(torch.int16)[total_words:nd * shard_size].zero_()
        t0.record()
        if scheme == "spec":
            _lib.call("kvec_rs16_pack", K_TN.data_ptr(), V_TN.data_ptr(), shards.data_ptr(),
                      T * n, T * n, _stream(shards))
        else:
            rdp_kernel.fused_backup_full_kv(K_TN, V_TN, shards, nd, int(shard_size), int(T), int(n),
                                            int(star_base))
    if scheme == "spec":
        rows = _rows_u8(shards)
        spec.rdp_encode(rows[:nd], rows[nd], rows[nd + 1], p, unit_bytes=spec.RDP_UNIT)
    t1.record()
    torch.cuda.synchronize()
    backup_ms = t0.elapsed_time(t1)
    return {
        "shards_KV": shards,
        "shard_size": int(shard_size),
        "seq_len": int(T),
        "n": int(n),
        "num_data_shards": nd,
        "star_base": int(star_base),
        "shape_BHTD": (B, H, T, D),
        "backup_ms": backup_ms,
        "pad_words": int(pad_words),
        "dtype": keys_bhtd.dtype,
        "scheme": scheme,
        "p": p,
    }


def fused_recovery_full_kv(pkg: dict, missing_a: int, missing_b: int = -1):
    """benchmark/rdp/main.py:95-126: returns (keys_bhtd, values_bhtd, stats).
    For a pkg of scheme "spec" the lost rows (data 0..nd-1, P = nd, Q = nd+1;
    other indices are ignored) are rebuilt by the textbook RDP decode first."""
    shards = pkg["shards_KV"]
    shard_size = pkg["shard_size"]
    T = pkg["seq_len"]
    n = pkg["n"]
    nd = pkg["num_data_shards"]
    star_base = pkg["star_base"]
    B, H, _, D = pkg["shape_BHTD"]
    dtype = pkg.get("dtype", torch.float16)

    is_spec = pkg.get("scheme", "ghostserve") == "spec"
    _lib.require_cuda(shards, what="fused_recovery_full_kv tensor")
    # the rows written straight to K and V when the layout allows it (known
    # before they are allocated: heads of whole 16 bytes, rows of 64 words and
    # more) and unless copies are faster; else, and where n is not the shape's,
    # through a token-major copy
    kv = None
    if (D * dtype.itemsize % 16 == 0 and (is_spec or shard_size >= 64) and n == B * H * D
            and not _copies_are_faster(B, H, T, D * dtype.itemsize)):
        kv_shape = (int(B), int(H), int(T), int(D))
        keys = torch.empty(kv_shape, dtype=dtype, device=shards.device)
        values = torch.empty(kv_shape, dtype=dtype, device=shards.device)
        kv = _lib.kv_bhtd(keys, values)
    t0 = torch.cuda.Event(enable_timing=True)
    t1 = torch.cuda.Event(enable_timing=True)
    t0.record()
    if is_spec:
        lost = [int(e) for e in (missing_a, missing_b) if 0 <= int(e) < nd + 2]
        spec.rdp_decode(_rows_u8(shards), int(pkg["p"]), lost, unit_bytes=spec.RDP_UNIT)
        direct = kv is not None and _lib.call_if_built(
            "kvec_kv_unpack_bhtd", shards.data_ptr(), 2 * int(nd) * int(shard_size), kv, _stream(shards))
    else:
        direct = kv is not None and _lib.call_if_built(
            "kvec_gs_rdp_recover_kv", shards.data_ptr(), kv, int(nd), int(shard_size), int(star_base),
            int(missing_a), int(missing_b), _stream(shards))
    if not direct:
        packed_TN = torch.empty(2 * T * n, dtype=dtype, device=shards.device)
        if is_spec:
            _lib.call("kvec_rs16_split", shards.data_ptr(), packed_TN.data_ptr(),
                      packed_TN[T * n:].data_ptr(), T * n, T * n, _stream(shards))
        else:
            rdp_kernel.fused_recovery_full_kv(shards, packed_TN, int(nd), int(shard_size), int(T),
                                              int(n), int(star_base), int(missing_a),
                                              int(missing_b))
    t1.record()
    torch.cuda.synchronize()
    recover_ms = t0.elapsed_time(t1)
    if not direct:
        keys, values = (x.view(T, B, H, D).permute(1, 2, 0, 3).contiguous()
                        for x in (packed_TN[:T * n], packed_TN[T * n:]))
    return keys, values, {"recover_ms": recover_ms}
