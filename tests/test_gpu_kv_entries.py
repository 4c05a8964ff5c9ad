"""The one-pass K/V entry points called directly, so that nothing else can have
made the bytes: every buffer they write lies between guard bytes, K and V may
have gaps that must stay, and the wrappers are held to the entry point that a
layout has."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

GUARD = 4096


class Guarded:
    """`n` bytes of GPU memory of 0xA5 between guards of the same."""

    def __init__(self, n, gpu):
        self.n = n
        self.all = torch.full((n + 2 * GUARD,), 0xA5, dtype=torch.uint8, device=gpu)
        self.b = self.all[GUARD:GUARD + n]

    def intact(self):
        a = self.all
        return bool((a[:GUARD] == 0xA5).all()) and bool((a[GUARD + self.n:] == 0xA5).all())


# memory order of [B, H, T, D] tensors: the dimensions outermost first, and the
# words between the end of a head and the next
ORDERS = {"head": ((0, 1, 2), 0), "token": ((0, 2, 1), 0), "pool": ((2, 0, 1), 0), "gaps": ((0, 1, 2), 24),
          "token gaps": ((0, 2, 1), 8)}


def _layout(order, B, H, T, D):
    """(words of the buffer, strides over B, H, T)."""
    dims, gap = ORDERS[order]
    n, st = D + gap, [0, 0, 0]
    for d in reversed(dims):
        st[d] = n
        n *= (B, H, T)[d]
    return n, st


class KV:
    """K and V of one layout, each guarded; words set from a seed."""

    def __init__(self, pkg, gpu, order, B, H, T, D, seed):
        n, st = _layout(order, B, H, T, D)
        self.buf = [Guarded(2 * n, gpu) for _ in range(2)]
        self.t = [b.b.view(torch.int16).as_strided((B, H, T, D), (*st, 1)) for b in self.buf]
        self.mask = torch.zeros(n, dtype=torch.bool, device=gpu)
        self.mask.as_strided((B, H, T, D), (*st, 1)).fill_(True)
        g = torch.Generator(device="cpu").manual_seed(seed)
        self.want = [torch.randint(-32768, 32768, (B, H, T, D), generator=g, dtype=torch.int16) for _ in range(2)]
        self.c = pkg._lib.KvBhtd(self.t[0].data_ptr(), self.t[1].data_ptr(), B, H, T, 2 * D, *(2 * s for s in st))

    def fill(self):
        for t, w in zip(self.t, self.want):
            t.copy_(w)

    def clear(self):
        for b in self.buf:
            b.all.fill_(0xA5)

    def written(self):
        """K and V hold their words, and nothing else was written."""
        fill = -23131   # 0xA5A5
        return all(b.intact() and torch.equal(t.cpu(), w) and bool((b.b.view(torch.int16)[~self.mask] == fill).all())
                   for b, t, w in zip(self.buf, self.t, self.want))

    def tn(self):
        return [w.permute(2, 0, 1, 3).contiguous().numpy().reshape(w.shape[2], -1).view(np.uint16) for w in self.want]

    def flat(self):
        return np.concatenate([w.numpy().reshape(-1).view(np.uint16) for w in self.want])


def _call(pkg, name, *args):
    L = pkg._lib.lib()
    rc = getattr(L, name)(*args, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, L.kvec_last_error()
    torch.cuda.synchronize()


def _bytes(x):
    return x.cpu().numpy()


@pytest.mark.parametrize("order", list(ORDERS))
@pytest.mark.parametrize("B,H,T,D,nd", [(2, 3, 37, 80, 1), (1, 8, 512, 128, 8), (3, 2, 101, 8, 5), (2, 4, 203, 64, 12),
                                        (4, 8, 521, 128, 6)])
def test_star_entries(pkg, ora, gpu, order, B, H, T, D, nd):
    kv = KV(pkg, gpu, order, B, H, T, D, T)
    kv.fill()
    want = ora.gs_backup(*kv.tn(), nd, 2)
    S = want.shape[1]
    sh = Guarded(want.nbytes, gpu)
    _call(pkg, "kvec_gs_rdp_backup_kv", kv.c, sh.b.data_ptr(), nd, S, 2)
    assert sh.intact() and np.array_equal(_bytes(sh.b), want.view(np.uint8).reshape(-1)) and kv.written()
    for lost in (-1, 0, nd - 1):
        if lost >= 0:
            sh.b.view(torch.int16).view(nd + 2, S)[lost] = 0x5A5A
        kv.clear()
        _call(pkg, "kvec_gs_rdp_recover_kv", sh.b.data_ptr(), kv.c, nd, S, 2, lost, -1)
        assert kv.written() and sh.intact() and np.array_equal(_bytes(sh.b), want.view(np.uint8).reshape(-1)), lost


@pytest.mark.parametrize("order", list(ORDERS))
@pytest.mark.parametrize("B,H,T,D,extra", [(2, 3, 37, 80, 0), (1, 8, 512, 128, 16), (3, 2, 101, 8, 4096 + 48), (1, 1, 1, 8, 0)])
def test_pack_entries(pkg, gpu, order, B, H, T, D, extra):
    kv = KV(pkg, gpu, order, B, H, T, D, T)
    kv.fill()
    flat = np.concatenate([x.reshape(-1) for x in kv.tn()]).view(np.uint8)
    rows = Guarded(flat.size + extra, gpu)
    _call(pkg, "kvec_kv_pack_bhtd", kv.c, rows.b.data_ptr(), rows.n)
    got = _bytes(rows.b)
    assert rows.intact() and np.array_equal(got[:flat.size], flat) and not got[flat.size:].any() and kv.written()
    kv.clear()
    rows.b[flat.size:] = 0x77   # padding, not the stream's
    _call(pkg, "kvec_kv_unpack_bhtd", rows.b.data_ptr(), rows.n, kv.c)
    assert kv.written() and rows.intact()


@pytest.mark.parametrize("spec", [False, True])
@pytest.mark.parametrize("k,m", [(1, 1), (5, 2), (8, 3), (10, 4), (16, 4)])
@pytest.mark.parametrize("B,H,T,D,more", [(2, 3, 101, 80, 0), (1, 8, 512, 128, 8), (1, 1, 2051, 8, 5)])
def test_rs_entries(pkg, ora, gpu, spec, k, m, B, H, T, D, more):
    """Rows of K || V and `more` words; GF(2^8) rows are whole 16 bytes."""
    kv = KV(pkg, gpu, "head", B, H, T, D, k)
    kv.fill()
    flat = kv.flat()
    S = -(-flat.size // k) + more
    S = -(-S // 8) * 8 if spec else S
    data = np.zeros(k * S, np.uint16)
    data[:flat.size] = flat
    if spec:
        rows = data.view(np.uint8).reshape(k, 2 * S)
        want = np.concatenate([rows.reshape(-1)] + [np.asarray(p).reshape(-1) for p in ora.rs8_encode([r.copy() for r in rows], m)])
    else:
        want = ora.rs16_encode(data, k, m, S, *pkg.rs.init_gf_tables()).view(np.uint8).reshape(-1)
    half, code, size = flat.nbytes // 2, ("rs8" if spec else "rs16"), (2 * S if spec else S)
    kp, vp = (t.data_ptr() for t in kv.t)
    sh = Guarded(want.nbytes, gpu)
    _call(pkg, f"kvec_{code}_encode_kv", kp, vp, half, sh.b.data_ptr(), k, m, size)
    assert sh.intact() and np.array_equal(_bytes(sh.b), want) and kv.written()
    for n in range(1, min(k, m) + 1):
        for lost in (np.arange(n, dtype=np.int32), np.arange(k - n, k, dtype=np.int32)):
            sh.b.view(k + m, 2 * S)[torch.from_numpy(lost).long().to(gpu)] = 0x5A
            kv.clear()
            _call(pkg, f"kvec_{code}_recover_kv", sh.b.data_ptr(), kp, vp, half, k, m, size, lost.ctypes.data, n)
            assert kv.written() and sh.intact() and np.array_equal(_bytes(sh.b), want), lost


# the wrappers take the entry point where there is one: (layout, rows) -> the
# answers of the backup and of the recovery, None: not asked
@pytest.mark.parametrize("scheme", ["ghostserve", "spec"])
@pytest.mark.parametrize("order,D,nd,backup,recovery", [
    ("head", 128, 8, True, True), ("token", 64, 5, True, True), ("gaps", 8, 12, True, True), ("head", 64, 13, None, True),
    ("head", 64, 17, None, False), ("head", 20, 5, None, None)])
def test_wrappers_take_the_entry_points(pkg, gpu, monkeypatch, scheme, order, D, nd, backup, recovery):
    if scheme == "spec":   # its rows are packed whatever their number, up to p = 13
        if nd > 12:
            pytest.skip("past p = 13")
    kv = KV(pkg, gpu, order, 1, 4, 257, D, nd)
    kv.fill()
    took = []
    real = pkg._lib.call_if_built
    monkeypatch.setattr(pkg._lib, "call_if_built", lambda name, *a: took.append(real(name, *a)) or took[-1])
    K, V = (t.view(torch.float16) for t in kv.t)
    pk = pkg.rdp.fused_backup_full_kv(K, V, nd, scheme=scheme)
    assert took == ([] if backup is None else [backup])
    took.clear()
    k2, v2, _ = pkg.rdp.fused_recovery_full_kv(pk, 0)
    assert took == ([] if recovery is None else [recovery])
    assert all(torch.equal(x.view(torch.int16).cpu(), w) for x, w in zip((k2, v2), kv.want))


@pytest.mark.parametrize("scheme,k,m,lost,encode,decode", [
    ("ghostserve", 6, 2, [1, 4], [True], [True]), ("ghostserve", 6, 5, [0], [False], [True]),
    ("ghostserve", 6, 2, [1, 6], [True], []), ("ghostserve", 6, 2, [], [True], []),
    ("ghostserve", 65, 2, [1], [True], [False]), ("spec", 6, 2, [1, 6], [True], [True]),
    ("spec", 8, 4, [0, 1, 2, 3], [True], [True]), ("spec", 6, 5, [0], [], []), ("spec", 33, 1, [], [], [])])
def test_rs_wrappers_take_the_entry_points(pkg, gpu, monkeypatch, scheme, k, m, lost, encode, decode):
    kv = KV(pkg, gpu, "head", 1, 4, 257, 64, k)
    kv.fill()
    took = []
    real = pkg._lib.call_if_built
    monkeypatch.setattr(pkg._lib, "call_if_built", lambda name, *a: took.append(real(name, *a)) or took[-1])
    K, V = (t.view(torch.float16) for t in kv.t)
    if k > 32 and scheme == "spec":   # past the GF(2^8) code's limits: refused by the general path
        with pytest.raises(pkg._lib.KvecError):
            pkg.rs.forward_encode_kv(K, V, k, m, scheme=scheme)
        assert took == encode
        return
    sh, meta = pkg.rs.forward_encode_kv(K, V, k, m, scheme=scheme)
    assert took == encode
    took.clear()
    for e in lost:
        sh.view(torch.int16)[e] = 0x5A5A
    k2, v2 = pkg.rs.backwards_decode_kv(sh, meta, lost)
    assert took == decode
    assert all(torch.equal(x.view(torch.int16).cpu(), w) for x, w in zip((k2, v2), kv.want))


# both sides of the lines past which many heads of 16 bytes are copied
@pytest.mark.parametrize("scheme", ["ghostserve", "spec"])
@pytest.mark.parametrize("order,B,H,T,took_backup,took_recovery", [
    ("head", 1, 192, 4556, True, True), ("head", 1, 192, 4560, None, None), ("head", 1, 191, 4600, True, True),
    ("head", 5, 64, 3001, None, None), ("token", 5, 64, 3001, True, None), ("pool", 5, 64, 3001, True, None),
    ("token", 200, 1, 4400, None, None), ("pool", 200, 1, 4400, True, None)])
def test_many_heads_of_16_bytes(pkg, ora, gpu, monkeypatch, scheme, order, B, H, T, took_backup, took_recovery):
    kv = KV(pkg, gpu, order, B, H, T, 8, T)
    kv.fill()
    took = []
    real = pkg._lib.call_if_built
    monkeypatch.setattr(pkg._lib, "call_if_built", lambda name, *a: took.append(real(name, *a)) or took[-1])
    pk = pkg.rdp.fused_backup_full_kv(*(t.view(torch.float16) for t in kv.t), 5, scheme=scheme)
    want = ora.gs_backup(*kv.tn(), 5, 0)
    if scheme == "ghostserve":
        assert np.array_equal(pk["shards_KV"].cpu().numpy(), want)
    pk["shards_KV"].view(torch.int16)[3] = 0x5A5A
    k2, v2, _ = pkg.rdp.fused_recovery_full_kv(pk, 3)
    assert took == [x for x in (took_backup, took_recovery) if x]
    assert all(torch.equal(x.view(torch.int16).cpu(), w) for x, w in zip((k2, v2), kv.want))


# row tensors just below 2 GiB, K and V of 0.8 GB: 32-bit offsets near their end
@pytest.mark.parametrize("H,D", [(1, 128), (8, 64)])
def test_star_entries_near_2gib(pkg, gpu, H, D):
    nd = 6
    S = ((1 << 30) // (nd + 2) - 64) // (nd * H * D) * nd * H * D   # words of a row; whole tokens in all rows
    T = nd * S // (2 * H * D)
    K, V = (torch.empty((1, H, T, D), dtype=torch.int16, device=gpu).random_() for _ in range(2))
    stream = torch.cat([x.permute(2, 0, 1, 3).reshape(-1) for x in (K, V)]).view(nd, S)
    pk = pkg.rdp.fused_backup_full_kv(K.view(torch.float16), V.view(torch.float16), nd, star_base=3)
    sh = pk["shards_KV"].view(torch.int16)
    assert sh.shape == (nd + 2, S) and sh.numel() * 2 < 1 << 31
    P, Q = torch.zeros_like(sh[0]), torch.zeros_like(sh[0])
    for r in range(nd):
        P ^= stream[r]
        x = torch.roll(stream[r], r)
        x[(3 + 2 * r) % S] = 0   # the star word's diagonal
        Q ^= x
    assert torch.equal(sh[:nd], stream) and torch.equal(sh[nd], P) and torch.equal(sh[nd + 1], Q)
    for lost in (0, nd - 1):
        sh[lost] = 0x5A5A
        k2, v2, _ = pkg.rdp.fused_recovery_full_kv(pk, lost)
        assert torch.equal(sh[:nd], stream)
        assert torch.equal(k2.view(torch.int16), K) and torch.equal(v2.view(torch.int16), V)


@pytest.mark.parametrize("scheme", ["ghostserve", "spec"])
@pytest.mark.parametrize("k,m,short", [(6, 2, 0), (6, 2, 3), (7, 4, 5)])
def test_rs_entries_near_2gib(pkg, gpu, scheme, k, m, short):
    S = (1 << 30) // (k + m) // 8 * 8 - 32 - (0 if scheme == "spec" else short)
    n = k * S // 2 // 8 * 8
    K, V = (torch.empty((1, 1, n // 8, 8), dtype=torch.int16, device=gpu).random_() for _ in range(2))
    sh, meta = pkg.rs.forward_encode_kv(K.view(torch.float16), V.view(torch.float16), k, m, scheme=scheme)
    S = meta["shard_sz"]
    assert sh.numel() * 2 < 1 << 31
    data = torch.zeros(k * S, dtype=torch.int16, device=gpu)
    data[:2 * n] = torch.cat([K.view(-1), V.view(-1)])
    assert torch.equal(sh.view(torch.int16)[:k].reshape(-1), data)
    par = torch.empty((k + m, S), dtype=torch.uint16, device=gpu)
    if scheme == "spec":
        rows, out = data.view(torch.uint8).view(k, -1), par.view(torch.uint8).view(k + m, -1)
        pkg.spec.rs8_encode([rows[i] for i in range(k)], [out[k + i] for i in range(m)])
    else:
        pkg.rs.rs_kernel.encode_rs_u16(data.view(torch.uint16), par, k, m, S, *pkg.rs.device_gf_tables(gpu))
    assert torch.equal(sh.view(torch.int16)[k:], par.view(torch.int16)[k:])
    for lost in (list(range(m)), [k - 1]):
        for e in lost:
            sh.view(torch.int16)[e] = 0x5A5A
        k2, v2 = pkg.rs.backwards_decode_kv(sh, meta, lost)
        assert torch.equal(sh.view(torch.int16)[:k].reshape(-1), data)
        assert torch.equal(k2.view(torch.int16), K) and torch.equal(v2.view(torch.int16), V)
