"""Backup, recovery and encode kernels that read and write K and V where they
lie, against the oracle on the permuted copies: strided tensors, every row
count, rows at every alignment, both tile widths, and the layouts that fall
back to the copies."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _kv(B, H, T, D, order, gpu, seed=0):
    """K and V indexed [B, H, T, D], random words, in the memory order given."""
    g = torch.Generator(device="cpu").manual_seed(seed + T)
    out = []
    for _ in range(2):
        x = torch.randint(-32768, 32768, (B, H, T, D), generator=g, dtype=torch.int16)
        if order == "token":       # [B, T, H, D] cache
            t = x.permute(0, 2, 1, 3).contiguous().to(gpu).permute(0, 2, 1, 3)
        elif order == "wide":      # heads of a wider tensor
            t = torch.zeros((B, H, T, D + 24), dtype=torch.int16, device=gpu)[..., 8:8 + D]
            t.copy_(x)
        elif order == "odd":       # two bytes past alignment
            buf = torch.zeros(x.numel() + 8, dtype=torch.int16, device=gpu)
            t = buf[1:1 + x.numel()].view(B, H, T, D)
            t.copy_(x)
        else:
            t = x.to(gpu)
        out.append(t.view(torch.float16))
    return out


def _tn(x):
    B, H, T, D = x.shape
    return x.view(torch.int16).permute(2, 0, 1, 3).contiguous().cpu().numpy().reshape(T, -1).view(np.uint16)


# nd 1..8 at word counts that leave rows at every alignment; 128-thread tiles
# (stripes of few tiles) and, for the last three, 512-thread ones; one row
# that is a whole number of tiles; D of 80 (10 chunks per head)
@pytest.mark.parametrize("B,H,T,D,nd", [
    (1, 8, 512, 128, 8), (2, 1, 33, 128, 6), (1, 2, 5, 64, 3), (3, 2, 17, 80, 7), (1, 1, 64, 128, 8),
    (2, 4, 101, 128, 5), (1, 1, 1024, 8, 4), (1, 3, 7, 16, 2), (4, 8, 263, 128, 1), (4, 8, 521, 128, 2),
    (8, 8, 800, 128, 6), (1, 2, 4096, 64, 1),
    # nine rows and more: two edge chunks; past twelve the backup copies first
    (1, 8, 512, 128, 9), (2, 3, 101, 80, 10), (1, 2, 37, 128, 12), (1, 2, 37, 128, 13), (2, 4, 203, 64, 16),
    (8, 8, 2053, 128, 10), (1, 1, 9, 64, 17)])
@pytest.mark.parametrize("order", ["head", "token", "wide", "odd"])
def test_gs_rdp_kv_layouts(pkg, ora, gpu, B, H, T, D, nd, order):
    K, V = _kv(B, H, T, D, order, gpu)
    sb = (B * T) % 5 - 1
    want = ora.gs_backup(_tn(K), _tn(V), nd, sb)
    pk = pkg.rdp.fused_backup_full_kv(K, V, nd, star_base=sb)
    assert np.array_equal(pk["shards_KV"].cpu().numpy(), want)
    S = pk["shard_size"]
    for a, b in [(-1, -1), (nd - 1, -1), (0, -1), (nd // 2, nd)]:
        sh = want.copy()
        if 0 <= a < nd:
            sh[a] = 0x5A5A
        exp = sh.copy()
        ora.gs_recover(exp, nd, S, sb, a, b)
        pk["shards_KV"] = torch.from_numpy(sh.view(np.int16)).to(gpu).view(torch.uint16)
        k2, v2, _ = pkg.rdp.fused_recovery_full_kv(pk, a, b)
        assert np.array_equal(pk["shards_KV"].cpu().numpy(), exp), (a, b)
        assert torch.equal(k2.view(torch.int16), K.view(torch.int16).contiguous()), (a, b)
        assert torch.equal(v2.view(torch.int16), V.view(torch.int16).contiguous()), (a, b)


# (k, m) with one to four parities (packed words and bit planes; five takes the
# pack and the general encode), rows of multiples of 16 bytes and not, odd and
# even k, rows under a tile, a whole number of tiles, tiles and 2-30 bytes,
# zero padding across several rows, stripes of many tiles
@pytest.mark.parametrize("k,m", [(4, 1), (5, 2), (6, 2), (1, 1), (5, 3), (8, 3), (10, 4), (16, 4), (3, 4), (17, 2),
                                 (6, 5)])
@pytest.mark.parametrize("B,H,T,D", [(1, 1, 40, 16), (1, 2, 33, 128), (2, 3, 101, 80), (1, 8, 256, 128),
                                     (1, 1, 2051, 8), (3, 4, 521, 128)])
def test_rs16_kv(pkg, ora, gpu, k, m, B, H, T, D):
    _rs16_round(pkg, ora, gpu, k, m, B, H, T, D)


# rows past 8 MiB, the other tile width of the decode
@pytest.mark.parametrize("k,m,T", [(2, 2, 8193), (1, 1, 4098), (3, 2, 12289)])
def test_rs16_kv_long_rows(pkg, ora, gpu, k, m, T):
    _rs16_round(pkg, ora, gpu, k, m, 1, 4, T, 128)


def _rs16_round(pkg, ora, gpu, k, m, B, H, T, D):
    K, V = _kv(B, H, T, D, "head", gpu, seed=k)
    sh, meta = pkg.rs.forward_encode_kv(K, V, k, m)
    S = meta["shard_sz"]
    data = np.zeros(k * S, np.uint16)
    flat = np.concatenate([x.view(torch.int16).cpu().numpy().reshape(-1).view(np.uint16) for x in (K, V)])
    data[:flat.size] = flat
    want = ora.rs16_encode(data, k, m, S, *pkg.rs.init_gf_tables())
    assert np.array_equal(sh.cpu().numpy(), want)
    # one to m lost rows, at both ends and adjacent; a lost parity row 0 (the
    # general reconstruct); every byte of the shards as encoded afterwards
    lost = [list(range(n)) for n in range(1, min(m, k) + 1)] + [list(range(k - n, k)) for n in range(1, min(m, k) + 1)]
    lost += [[0, k - 1], [k // 2]] if m > 1 and k > 1 else []
    lost += [[k // 2, k]] if m > 1 else []
    full = sh.clone()
    for er in lost:
        sh.copy_(full)
        for e in er:
            if e < k:
                sh.view(torch.int16)[e] = 0x5A5A
        k2, v2 = pkg.rs.backwards_decode_kv(sh, meta, er)
        assert torch.equal(sh.view(torch.int16), full.view(torch.int16)), er
        assert torch.equal(k2.view(torch.int16), K.view(torch.int16)), er
        assert torch.equal(v2.view(torch.int16), V.view(torch.int16)), er


# GF(2^8) codes behind the same wrappers: one to four outputs in one pass (five
# parities: the pack and the shard kernels), odd and even k, rows of one chunk,
# a tile, tiles and a remainder; every parity row and mixes of lost rows
@pytest.mark.parametrize("k,m", [(1, 1), (4, 1), (5, 3), (6, 2), (8, 4), (10, 4), (16, 2), (9, 3), (6, 5)])
@pytest.mark.parametrize("B,H,T,D", [(1, 1, 9, 8), (1, 2, 33, 128), (2, 3, 101, 80), (1, 8, 512, 128), (3, 4, 521, 128)])
def test_rs8_kv(pkg, ora, gpu, k, m, B, H, T, D):
    K, V = _kv(B, H, T, D, "head", gpu, seed=k)
    sh, meta = pkg.rs.forward_encode_kv(K, V, k, m, scheme="spec")
    S = meta["shard_sz"]
    data = np.zeros(k * S, np.uint16)
    flat = np.concatenate([x.view(torch.int16).cpu().numpy().reshape(-1).view(np.uint16) for x in (K, V)])
    data[:flat.size] = flat
    rows = data.view(np.uint8).reshape(k, 2 * S)
    par = ora.rs8_encode([r.copy() for r in rows], m)
    want = np.concatenate([rows.reshape(-1)] + [np.asarray(p).reshape(-1) for p in par])
    assert np.array_equal(sh.cpu().numpy().view(np.uint8).reshape(-1), want)
    full = sh.clone()
    lost = [[e] for e in range(k + m)] + [list(range(min(m, k))), list(range(k + m - m, k + m))]
    lost += [[0, k + m - 1], [k - 1, k]] if m > 1 else []
    for er in lost:
        sh.copy_(full)
        for e in er:
            sh.view(torch.int16)[e] = 0x5A5A
        k2, v2 = pkg.rs.backwards_decode_kv(sh, meta, er)
        assert torch.equal(sh.view(torch.int16), full.view(torch.int16)), er
        assert torch.equal(k2.view(torch.int16), K.view(torch.int16)), er
        assert torch.equal(v2.view(torch.int16), V.view(torch.int16)), er


# separate shards of the shapes without a straight-line kernel: groups of four
# outputs and a remainder, odd and even input counts, shards of one chunk, a
# tile, a tile and a chunk
@pytest.mark.parametrize("k,m", [(8, 3), (8, 4), (6, 3), (12, 4), (16, 2), (8, 8), (9, 7), (32, 2), (1, 1), (3, 2)])
@pytest.mark.parametrize("S", [16, 8192, 8192 * 2 + 16, 70000])
def test_rs8_loop_shapes(pkg, ora, gpu, k, m, S):
    rng = np.random.default_rng(k * 10 + m)
    data = [rng.integers(0, 256, S, dtype=np.uint8) for _ in range(k)]
    par = [np.asarray(p).reshape(-1) for p in ora.rs8_encode(data, m)]
    want = [torch.from_numpy(x.copy()).to(gpu) for x in data + par]
    sh = [w.clone() for w in want]
    for p in sh[k:]:
        p.zero_()
    pkg.spec.rs8_encode(sh[:k], sh[k:])
    assert all(torch.equal(a, b) for a, b in zip(sh, want))
    for er in ([0], list(range(min(k, m))), list(range(k + m - m, k + m)), sorted({0, k + m - 1} if m > 1 else {k})):
        for e in er:
            sh[e].fill_(0x5A)
        pkg.spec.rs8_decode(sh, k, er)
        assert all(torch.equal(a, b) for a, b in zip(sh, want)), er


# both sides of the size from which two outputs of four to six inputs are coded
# straight-line
@pytest.mark.parametrize("k", [4, 5, 6])
@pytest.mark.parametrize("S", [(60 << 20) - 16, 60 << 20, (60 << 20) + 1040])
def test_rs8_straight_line_sizes(pkg, ora, gpu, k, S):
    g = torch.Generator(device=gpu).manual_seed(k)
    data = [torch.randint(-2**62, 2**62, (S // 8,), generator=g, device=gpu).view(torch.uint8) for _ in range(k)]
    par = [torch.empty_like(d) for d in data[:2]]
    pkg.spec.rs8_encode(data, par)
    at = torch.cat([torch.arange(0, 16 * 1024), torch.arange(S - 16 * 1024, S)]).to(gpu)
    want = ora.rs8_encode([d[at].cpu().numpy() for d in data], 2)
    assert all(np.array_equal(p[at].cpu().numpy(), np.asarray(w).reshape(-1)) for p, w in zip(par, want))
    full = [d.clone() for d in data[:2]]
    data[0].zero_()
    data[1].zero_()
    pkg.spec.rs8_decode(data + par, k, [0, 1])
    assert torch.equal(data[0], full[0]) and torch.equal(data[1], full[1])


# the same of the other shapes coded straight-line, one window a thread (8, 2)
# and two
@pytest.mark.parametrize("k,m,S", [(k, m, (mib << 20) + d) for k, m, mib in ((8, 2, 40), (10, 1, 48))
                                   for d in (-16, 0, 1040)])
def test_rs8_straight_line_wide(pkg, ora, gpu, k, m, S):
    g = torch.Generator(device=gpu).manual_seed(k)
    data = [torch.randint(-2**62, 2**62, (S // 8,), generator=g, device=gpu).view(torch.uint8) for _ in range(k)]
    par = [torch.empty_like(d) for d in data[:m]]
    pkg.spec.rs8_encode(data, par)
    at = torch.cat([torch.arange(0, 16 * 1024), torch.arange(S - 16 * 1024, S)]).to(gpu)
    want = ora.rs8_encode([d[at].cpu().numpy() for d in data], m)
    assert all(np.array_equal(p[at].cpu().numpy(), np.asarray(w).reshape(-1)) for p, w in zip(par, want))
    full = [d.clone() for d in data[:m]]
    for d in data[:m]:
        d.zero_()
    pkg.spec.rs8_decode(data + par, k, list(range(m)))
    assert all(torch.equal(a, b) for a, b in zip(data, full))


# P and Q of rows in place, nine to sixteen of them: every word alignment of the
# tensor, rows of exactly a tile, odd lengths, star words in the wrapped part
@pytest.mark.parametrize("nd", range(9, 17))
@pytest.mark.parametrize("soff,S,sb", [(0, 1024, 0), (3, 4096, -1), (5, 6149, 4090), (0, 64, 3), (7, 20481, 2),
                                       (1, 65, 60), (6, 530003, 0)])
def test_gs_parity_wide(pkg, ora, gpu, nd, soff, S, sb):
    rng = np.random.default_rng(nd + S)
    rows = rng.integers(0, 65536, (nd + 2, S), dtype=np.uint16)
    want = rows.copy()
    ora.gs_parity(want, nd, S, sb)
    buf = torch.full(((nd + 2) * S + 32,), 0x3C3C, dtype=torch.int16, device=gpu)
    buf[soff:soff + rows.size] = torch.from_numpy(rows.reshape(-1).view(np.int16)).to(gpu)
    pkg.rdp_kv_ops.compute_rdp_parity(buf.view(torch.uint16)[soff:soff + rows.size].view(nd + 2, S), nd, S, sb)
    got = buf.cpu().numpy().view(np.uint16)
    assert np.array_equal(got[soff:soff + rows.size], want.reshape(-1))
    assert (np.concatenate([got[:soff], got[soff + rows.size:]]) == 0x3C3C).all()


# the spec scheme's layout step from and to strided K and V
@pytest.mark.parametrize("B,H,T,D,nd", [(1, 8, 512, 128, 8), (3, 2, 17, 80, 5), (2, 4, 1301, 128, 6), (1, 1, 5, 8, 2)])
@pytest.mark.parametrize("order", ["head", "token", "wide", "odd"])
def test_rdp_spec_kv_layouts(pkg, ora, gpu, B, H, T, D, nd, order):
    K, V = _kv(B, H, T, D, order, gpu)
    pk = pkg.rdp.fused_backup_full_kv(K, V, nd, scheme="spec")
    S, n = pk["shard_size"], 2 * B * H * T * D
    flat = np.zeros(nd * S, np.uint16)
    flat[:n] = np.concatenate([_tn(K).reshape(-1), _tn(V).reshape(-1)])
    rows = flat.view(np.uint8).reshape(nd, 2 * S)
    Pw, Qw = ora.rdp_encode([r.copy() for r in rows], pk["p"], unit=pkg.spec.RDP_UNIT)
    got = pk["shards_KV"].cpu().numpy().view(np.uint8)
    assert np.array_equal(got[:nd], rows)
    assert np.array_equal(got[nd], Pw.reshape(-1)) and np.array_equal(got[nd + 1], Qw.reshape(-1))
    pk["shards_KV"].view(torch.int16)[nd - 1] = 0x5A5A
    pk["shards_KV"].view(torch.int16)[0] = 0x5A5A
    k2, v2, _ = pkg.rdp.fused_recovery_full_kv(pk, 0, nd - 1)
    assert np.array_equal(pk["shards_KV"].cpu().numpy().view(np.uint8), got)
    assert torch.equal(k2.view(torch.int16), K.view(torch.int16).contiguous())
    assert torch.equal(v2.view(torch.int16), V.view(torch.int16).contiguous())


@pytest.mark.parametrize("scheme", ["ghostserve", "spec"])
def test_rs_kv_graph_replay(pkg, gpu, scheme):
    """The one-pass encode and decode captured in one graph: every replay on
    fresh K and V, with eager calls between replays, gives the eager bytes."""
    k, m, lost = 6, 2, [1, 4]
    K, V = _kv(2, 4, 203, 128, "head", gpu)
    full, meta = pkg.rs.forward_encode_kv(K, V, k, m, scheme=scheme)   # tables and library loaded

    def step():
        sh, _ = pkg.rs.forward_encode_kv(K, V, k, m, scheme=scheme)
        before = sh.clone()
        for e in lost:
            sh.view(torch.int16)[e].fill_(0x5A5A)
        return before, sh, *pkg.rs.backwards_decode_kv(sh, meta, lost)

    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step()
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        before, sh, k2, v2 = step()
    for i in range(4):
        x, y = _kv(2, 4, 203, 128, "head", gpu, seed=100 + i)
        K.copy_(x)
        V.copy_(y)
        want, _ = pkg.rs.forward_encode_kv(x, y, k, m, scheme=scheme)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(before.view(torch.int16), want.view(torch.int16)), i
        assert torch.equal(sh.view(torch.int16), want.view(torch.int16)), i
        assert torch.equal(k2.view(torch.int16), x.view(torch.int16)), i
        assert torch.equal(v2.view(torch.int16), y.view(torch.int16)), i


@pytest.mark.parametrize("scheme", ["ghostserve", "spec"])
def test_rs_encode_refuses_host_values(pkg, gpu, monkeypatch, scheme):
    """V in host memory is refused before any entry point is asked (none is
    reached here either way: the stand-in fails the test)."""
    K, V = _kv(1, 2, 33, 128, "head", gpu)

    def asked(name, *args):
        pytest.fail(f"{name} was given a host pointer")

    monkeypatch.setattr(pkg._lib, "call_if_built", asked)
    with pytest.raises(ValueError, match="GPU"):
        pkg.rs.forward_encode_kv(K, V.cpu(), 6, 2, scheme=scheme)


@pytest.mark.parametrize("scheme", ["ghostserve", "spec"])
def test_rs_encode_of_shared_memory(pkg, gpu, scheme):
    """K and V are only read: the same tensor, or two views of one buffer that
    overlap, code like copies of them."""
    buf = torch.randint(-32768, 32768, (3 * 33 * 128,), dtype=torch.int16, device=gpu).view(torch.float16)
    K = buf[:2 * 33 * 128].view(1, 2, 33, 128)
    for V in (K, buf[33 * 128:].view(1, 2, 33, 128)):
        got, meta = pkg.rs.forward_encode_kv(K, V, 6, 2, scheme=scheme)
        want, _ = pkg.rs.forward_encode_kv(K.clone(), V.clone(), 6, 2, scheme=scheme)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
        k2, v2 = pkg.rs.backwards_decode_kv(got, meta, [0, 3])
        assert torch.equal(k2.view(torch.int16), K.view(torch.int16))
        assert torch.equal(v2.view(torch.int16), V.view(torch.int16))


def _packed_backup(pkg, gpu, nd, S, sb, tail):
    """K, V and the row tensor of the packed backup of nd rows of S words, the
    last `tail` of them padding (left as they were)."""
    n = nd * S - tail
    assert n % 16 == 0
    K, V = (torch.empty(n // 2, dtype=torch.int16, device=gpu).random_() for _ in range(2))
    sh = torch.zeros((nd + 2, S), dtype=torch.int16, device=gpu)
    pkg.rdp.rdp_kernel.fused_backup_full_kv(K.view(torch.float16).view(1, -1), V.view(torch.float16).view(1, -1),
                                            sh.view(torch.uint16), nd, S, 1, n // 2, sb)
    return K, V, sh


# both sides of the row length from which nine to sixteen rows are coded as they
# are packed, in one launch
@pytest.mark.parametrize("nd,S", [(9, (11 << 19) - 16), (9, 11 << 19), (10, (11 << 19) + 16), (11, (17 << 19) - 16),
                                  (16, 17 << 19)])
def test_packed_backup_row_lengths(pkg, ora, gpu, nd, S):
    K, V, sh = _packed_backup(pkg, gpu, nd, S, 3, 16)
    want = np.zeros((nd + 2, S), np.uint16)
    ora.gs_pack(*(x.cpu().numpy().view(np.uint16).reshape(1, -1) for x in (K, V)), want, nd, S, 1, K.numel())
    ora.gs_parity(want, nd, S, 3)
    assert np.array_equal(sh.cpu().numpy().view(np.uint16), want)


# a row tensor past 2 GiB
@pytest.mark.parametrize("nd", [9, 16])
def test_packed_backup_past_2gib(pkg, gpu, nd):
    S = ((1 << 30) // (nd + 2) // 16 + 1) * 16
    free, _ = torch.cuda.mem_get_info(gpu)
    if free < 24 << 30:
        pytest.skip("needs 24 GiB of free device memory")
    K, V, sh = _packed_backup(pkg, gpu, nd, S, 5, 0)
    assert torch.equal(sh[:nd].reshape(-1), torch.cat([K, V]))
    P, Q = torch.zeros_like(sh[0]), torch.zeros_like(sh[0])
    for r in range(nd):
        P ^= sh[r]
        x = torch.roll(sh[r], r)
        x[(5 + r + r) % S] = 0   # the star word's diagonal
        Q ^= x
    assert torch.equal(sh[nd], P) and torch.equal(sh[nd + 1], Q)


@pytest.mark.parametrize("scheme", ["ghostserve", "spec"])
@pytest.mark.parametrize("B,H,T,D,order,nd", [(1, 8, 33, 20, "head", 5), (2, 2, 65, 12, "token", 5),
                                              (1, 2, 33, 64, "odd", 5), (1, 1, 4, 20, "head", 5)])
def test_copied_layouts_ask_no_entry_point(pkg, gpu, monkeypatch, scheme, B, H, T, D, order, nd):
    """Layouts that no one-pass entry point takes go to the copies without
    preparing for one: heads of no whole 16 bytes, and K and V off alignment
    (whose recovery, into K and V of its own, is direct)."""
    K, V = _kv(B, H, T, D, order, gpu)
    asked = []
    real = pkg._lib.call_if_built
    monkeypatch.setattr(pkg._lib, "call_if_built", lambda name, *a: asked.append(name) or real(name, *a))
    pk = pkg.rdp.fused_backup_full_kv(K, V, nd, scheme=scheme)
    assert not asked
    k2, v2, _ = pkg.rdp.fused_recovery_full_kv(pk, 1)
    assert len(asked) == (order == "odd")
    assert torch.equal(k2.view(torch.int16), K.view(torch.int16).contiguous())
    assert torch.equal(v2.view(torch.int16), V.view(torch.int16).contiguous())


@pytest.mark.parametrize("as_given", [
    lambda er, gpu: torch.tensor(er, device=gpu), lambda er, gpu: list(torch.tensor(er, device=gpu)),
    lambda er, gpu: np.array(er), lambda er, gpu: tuple(er)], ids=["gpu tensor", "gpu scalars", "numpy", "tuple"])
def test_rs16_lost_rows_as_given(pkg, gpu, as_given):
    """The lost rows as a program may hold them."""
    K, V = _kv(1, 2, 33, 128, "head", gpu)
    sh, meta = pkg.rs.forward_encode_kv(K, V, 6, 2)
    for er in ([3], [1, 4]):
        for e in er:
            sh.view(torch.int16)[e] = 0x5A5A
        k2, v2 = pkg.rs.backwards_decode_kv(sh, meta, as_given(er, gpu))
        assert torch.equal(k2.view(torch.int16), K.view(torch.int16)), er
        assert torch.equal(v2.view(torch.int16), V.view(torch.int16)), er


def test_rs_decode_of_fewer_rows(pkg, gpu, monkeypatch):
    """A shard tensor without all the parity rows: the one-pass decode is told
    the rows that are there, or not asked.  (The stand-in launches nothing.)"""
    K, V = _kv(1, 2, 33, 128, "head", gpu)
    k, m = 6, 3

    class Asked(Exception):
        pass

    def asked(name, *args):
        raise Asked(name, args)

    for scheme in ("ghostserve", "spec"):
        sh, meta = pkg.rs.forward_encode_kv(K, V, k, m, scheme=scheme)
        for rows, lost in ((k + 1, [2]), (k + 2, [0, 5])):
            with monkeypatch.context() as mp:
                mp.setattr(pkg._lib, "call_if_built", asked)
                mp.setattr(pkg.spec, "rs8_decode", lambda *a: asked("general", *a))
                # (the general decode of scheme "spec" refuses such a tensor when its
                # bytes do not make k + m equal rows)
                with pytest.raises((Asked, RuntimeError)) as e:
                    pkg.rs.backwards_decode_kv(sh[:rows].clone(), meta, lost)
            if scheme == "spec":
                assert e.type is RuntimeError or e.value.args[0] == "general"
            else:
                name, args = e.value.args
                assert name == "kvec_rs16_recover_kv" and args[4] + args[5] == rows
                part = sh[:rows].clone()
                part.view(torch.int16)[lost] = 0x5A5A
                k2, v2 = pkg.rs.backwards_decode_kv(part, meta, lost)
                assert torch.equal(part.view(torch.int16), sh[:rows].view(torch.int16))
                assert torch.equal(k2.view(torch.int16), K.view(torch.int16))
                assert torch.equal(v2.view(torch.int16), V.view(torch.int16))


@pytest.mark.parametrize("scheme", ["ghostserve", "spec"])
def test_rdp_recovery_refuses_other_shape(pkg, gpu, scheme):
    """A package whose words a token are not its shape's."""
    K, V = _kv(1, 4, 65, 64, "head", gpu)
    pk = pkg.rdp.fused_backup_full_kv(K, V, 5, scheme=scheme)
    for shape in ((1, 2, 65, 64), (1, 4, 65, 32)):
        with pytest.raises(RuntimeError):
            pkg.rdp.fused_recovery_full_kv(dict(pk, shape_BHTD=shape), 1)


# three and four parities around the lines past which many short rows of whole
# 8 KiB are packed and coded apart: (k, m, bytes of a row, one pass)
@pytest.mark.parametrize("k,m,Sb,one_pass", [
    (27, 3, 8192, True), (28, 3, 8192, False), (32, 3, 8192 + 16, True), (39, 4, 16384, True), (40, 4, 16384, False),
    (40, 4, 256 << 10, True), (64, 4, 256 << 10, False), (64, 4, 1 << 20, True), (96, 3, (1 << 20) + 8192, False),
    (30, 3, 1536 << 10, True), (64, 2, 8192, True)])
def test_rs16_many_short_rows(pkg, ora, gpu, monkeypatch, k, m, Sb, one_pass):
    T = k * Sb // 512   # K and V of one head of 128
    K, V = _kv(1, 1, T, 128, "head", gpu, seed=k)
    took = []
    real = pkg._lib.call_if_built
    monkeypatch.setattr(pkg._lib, "call_if_built", lambda name, *a: took.append(real(name, *a)) or took[-1])
    sh, meta = pkg.rs.forward_encode_kv(K, V, k, m)
    assert meta["shard_sz"] * 2 == Sb and took == [one_pass]
    data = np.zeros(k * meta["shard_sz"], np.uint16)
    flat = np.concatenate([x.view(torch.int16).cpu().numpy().reshape(-1).view(np.uint16) for x in (K, V)])
    data[:flat.size] = flat
    want = ora.rs16_encode(data, k, m, meta["shard_sz"], *pkg.rs.init_gf_tables())
    assert np.array_equal(sh.cpu().numpy(), want)
