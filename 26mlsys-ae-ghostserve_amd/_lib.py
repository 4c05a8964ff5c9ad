"""ctypes binding of libkvec.so (the C ABI declared in include/kvec.h).

torch is imported before the library is opened on purpose: torch ships its own
HIP runtime with the same soname (libamdhip64.so.7), and opening libkvec after
torch makes the dynamic linker bind libkvec to that same runtime, so the
hipStream_t handles torch hands out are valid inside libkvec.

There is no fallback: if libkvec.so is missing or fails to load, every entry
point raises.
"""
from __future__ import annotations

import ctypes as C
import os

import torch  # noqa: F401  (must precede CDLL, see module docstring)

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libkvec.so")

# torch's own accessor of a stream handle; not public, so maybe not there
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)

_vp = C.c_void_p
_i = C.c_int
_i64 = C.c_int64
_pp = C.POINTER(C.c_void_p)

class PagedKV(C.Structure):
    """struct kvec_paged_kv of include/kvec.h."""
    _fields_ = [
        ("pool", C.c_void_p),
        ("pool_pages", C.c_int64),
        ("layers", C.c_int),
        ("token_bytes", C.c_int64),
        ("page_tokens", C.c_int),
        ("page_table", C.c_void_p),
        ("batch", C.c_int),
        ("pages_per_seq", C.c_int),
        ("tok_off", C.c_int),
        ("tokens", C.c_int),
    ]


_kvp = C.POINTER(PagedKV)


class ChunkStripe(C.Structure):
    """struct kvec_chunk_stripe of include/kvec.h."""
    _fields_ = [
        ("data", C.POINTER(C.c_void_p)),
        ("k", C.c_int),
        ("P", C.c_void_p),
        ("Q", C.c_void_p),
        ("p", C.c_int),
        ("rs", C.POINTER(C.c_void_p)),
        ("m", C.c_int),
        ("row_bytes", C.c_int64),
        ("region_off", C.c_int64),
        ("width", C.c_int64),
        ("unit_bytes", C.c_int64),
    ]


_csp = C.POINTER(ChunkStripe)


class KvBhtd(C.Structure):
    """struct kvec_kv_bhtd of include/kvec.h."""
    _fields_ = [
        ("k", C.c_void_p),
        ("v", C.c_void_p),
        ("B", C.c_int64),
        ("H", C.c_int64),
        ("T", C.c_int64),
        ("head_bytes", C.c_int64),
        ("stride_b", C.c_int64),
        ("stride_h", C.c_int64),
        ("stride_t", C.c_int64),
    ]


_kbp = C.POINTER(KvBhtd)

# name -> (restype, argtypes); mirrors include/kvec.h
SIGNATURES = {
    "kvec_version": (_i, []),
    "kvec_strerror": (C.c_char_p, [_i]),
    "kvec_last_error": (C.c_char_p, []),
    "kvec_rdp_encode": (_i, [_pp, _i, _vp, _vp, _i, _i64, _i64, _vp]),
    "kvec_rdp_decode": (_i, [_pp, _i, _i, _i64, _i64, _i, _i, _vp]),
    "kvec_rdp_row_bytes": (_i64, [_i64, _i, _i, _i64]),
    "kvec_rs8_cauchy": (_i, [_i, _i, _vp]),
    "kvec_rs8_encode": (_i, [_pp, _i, _pp, _i, _i64, _vp]),
    "kvec_rs8_decode": (_i, [_pp, _i, _i, _i64, _vp, _i, _vp]),
    "kvec_rs8_encode_kv": (_i, [_vp, _vp, _i64, _vp, _i, _i, _i64, _vp]),
    "kvec_rs8_recover_kv": (_i, [_vp, _vp, _vp, _i64, _i, _i, _i64, _vp, _i, _vp]),
    "kvec_kv_stream_bytes": (_i64, [_kvp]),
    "kvec_kv_gather": (_i, [_kvp, _vp, _vp]),
    "kvec_kv_gather_split": (_i, [_kvp, _vp, _vp, _vp]),
    "kvec_kv_scatter": (_i, [_kvp, _vp, _vp, _vp]),
    "kvec_rdp_encode_paged": (_i, [_kvp, _pp, _i, _vp, _vp, _i, _i64, _i64, _vp]),
    "kvec_rdp_decode_paged": (_i, [_kvp, _vp, _pp, _i, _vp, _vp, _i, _i64, _i64, _i, _i, _vp]),
    "kvec_chunk_width": (_i64, [_i64, _i, _i, _i64]),
    "kvec_chunk_encode_paged": (_i, [_kvp, _csp, _vp]),
    "kvec_chunk_decode_paged": (_i, [_kvp, _vp, _csp, _vp, _i, _vp]),
    "kvec_xor_encode": (_i, [_vp, _vp, _i, _i64, _vp]),
    "kvec_xor_encode_kv": (_i, [_vp, _vp, _i64, _vp, _i, _i64, _vp]),
    "kvec_xor_recover_kv": (_i, [_vp, _vp, _i, _i64, _i64, _i, _vp]),
    "kvec_xor_reconstruct": (_i, [_vp, _vp, _vp, _i64, _i, _vp, _i, _vp]),
    "kvec_pack_kv": (_i, [_vp, _vp, _vp, _i, _i, _vp]),
    "kvec_unpack_kv": (_i, [_vp, _vp, _i, _i, _vp]),
    "kvec_gs_rdp_backup": (_i, [_vp, _vp, _vp, _i, _i, _i, _i, _i, _vp]),
    "kvec_gs_rdp_recover": (_i, [_vp, _vp, _i, _i, _i, _i, _i, _i, _i, _vp]),
    "kvec_gs_rdp_backup_kv": (_i, [_kbp, _vp, _i, _i, _i, _vp]),
    "kvec_gs_rdp_recover_kv": (_i, [_vp, _kbp, _i, _i, _i, _i, _i, _vp]),
    "kvec_kv_pack_bhtd": (_i, [_kbp, _vp, _i64, _vp]),
    "kvec_kv_unpack_bhtd": (_i, [_vp, _i64, _kbp, _vp]),
    "kvec_gs_pack_row": (_i, [_vp, _vp, _vp, _i64, _i, _i64, _vp]),
    "kvec_gs_rdp_parity": (_i, [_vp, _i, _i, _i, _vp]),
    "kvec_hook_step": (_i, [_kvp, _vp, _vp, _i, _i, _i, _i, _vp, _vp, _vp, _vp, _pp]),
    "kvec_rs16_pack": (_i, [_vp, _vp, _vp, _i64, _i64, _vp]),
    "kvec_rs16_split": (_i, [_vp, _vp, _vp, _i64, _i64, _vp]),
    "kvec_rs16_encode": (_i, [_vp, _vp, _i, _i, _i, _vp, _vp, _vp]),
    "kvec_rs16_encode_kv": (_i, [_vp, _vp, _i64, _vp, _i, _i, _i, _vp]),
    "kvec_rs16_recover_kv": (_i, [_vp, _vp, _vp, _i64, _i, _i, _i, _vp, _i, _vp]),
    "kvec_rs16_reconstruct": (_i, [_vp, _i, _i, _i, _vp, _i, _vp, _vp, _vp, _vp]),
    "kvec_gf16_tables": (_i, [_vp, _vp]),
}

# major number of the include/kvec.h these signatures mirror (KVEC_VERSION / 10000)
ABI_MAJOR = 1

_lib = None


class KvecError(RuntimeError):
    """A libkvec call returned a non-zero status."""


def lib():
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(
                f"{LIB_PATH} is not built; run __graft_entry__.build() (hipcc, gfx950)")
        L = C.CDLL(LIB_PATH)
        for name, (res, args) in SIGNATURES.items():
            f = getattr(L, name)
            f.restype = res
            f.argtypes = args
        ver = L.kvec_version()
        if ver // 10000 != ABI_MAJOR:
            raise RuntimeError(f"{LIB_PATH} has ABI version {ver}; these bindings need major "
                               f"version {ABI_MAJOR} (rebuild with __graft_entry__.build())")
        _lib = L
    return _lib


def call(name: str, *args) -> int:
    rc = getattr(lib(), name)(*args)
    if rc != 0:
        msg = lib().kvec_last_error().decode(errors="replace")
        raise KvecError(f"{name} failed ({lib().kvec_strerror(rc).decode()}): {msg}")
    return rc


EUNSUPPORTED = -2


def call_if_built(name: str, *args) -> bool:
    """`call`, returning False instead of raising when the entry point does not
    take the layout (KVEC_EUNSUPPORTED: nothing was enqueued)."""
    rc = getattr(lib(), name)(*args)
    if rc == EUNSUPPORTED:
        return False
    if rc != 0:
        msg = lib().kvec_last_error().decode(errors="replace")
        raise KvecError(f"{name} failed ({lib().kvec_strerror(rc).decode()}): {msg}")
    return True


def kv_bhtd(k, v):
    """The kvec_kv_bhtd of K and V tensors indexed [B, H, T, D], or None when
    they differ in strides, a head's values are not adjacent, or heads or
    tensors do not start and end on 16 bytes (no entry point takes those)."""
    B, H, T, D = k.shape
    ks, vs = k.stride(), v.stride()
    es = k.element_size()
    kp, vp = k.data_ptr(), v.data_ptr()
    if ks != vs or ks[3] != 1 or (kp | vp | D * es) & 15:
        return None
    return KvBhtd(kp, vp, B, H, T, D * es, ks[0] * es, ks[1] * es, ks[2] * es)


def ptr_array(tensors) -> C.Array:
    return (C.c_void_p * len(tensors))(*[int(t.data_ptr()) for t in tensors])


def stream_handle(device) -> int:
    """hipStream_t of torch's current stream on ``device``.  For a GPU tensor's
    device it is read without building a Stream object: a small call is bound
    by its host time."""
    if (_raw_stream is not None and isinstance(device, torch.device) and device.type == "cuda"
            and device.index is not None):
        return _raw_stream(device.index)
    return int(torch.cuda.current_stream(device).cuda_stream)


def require_cuda(*tensors, what: str = "tensor") -> None:
    for t in tensors:
        if not t.is_cuda:
            raise ValueError(f"{what} must be a GPU (HIP) tensor")
        if not t.is_contiguous():
            raise ValueError(f"{what} must be contiguous")
