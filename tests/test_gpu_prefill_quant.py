"""Prefill over quantized caches on the matrix cores against the f64 oracle and
against the VALU kernel, at the edges of its tiles (128 rows per CTA, 32-key
blocks), with and without key splits, and over value ranges that f16 cannot hold
unscaled. The path holds its operands as pairs of f16 values (2^-22 relative) and
sums in f32, so the tolerance is that of f32 sums:
relative error (2-norm) 3e-6 = 2^-22 for each of q, K and p * V added up, plus the
roundings of sums over at most a few thousand terms (2^-24 sqrt(4000) = 4e-6 of a
single term, averaged over the row's independent dims)."""
import numpy as np
import pytest

from gpu_util import to_dev

pytestmark = pytest.mark.gpu
REL = 3e-6
PAIRS = [(kt, vt) for kt in range(1, 6) for vt in range(1, 6) if (kt, vt) != (1, 1)]


def rows_of(orc, t, n, nkv, seed, scale=1.0):
    x = orc.randn(n * nkv * 256, seed).reshape(n, nkv, 256) * np.float32(scale)
    x[:, :, 7] *= 8
    return orc.store_rows(t, x.ravel())


def run(rd4, torch, dev, q, k, v, pos0, nh, nkv, kt, vt, gate=None):
    out = torch.full(q.shape, float("nan"), dtype=torch.float32, device=dev)
    g = None if gate is None else to_dev(gate, torch, dev)
    rd4.prefill(to_dev(q, torch, dev), to_dev(k, torch, dev), to_dev(v, torch, dev), out, pos0, nh, nkv, 256,
                1 / 16, kt, vt, gate=g)
    torch.cuda.synchronize()
    return out.cpu().numpy(), None if g is None else g.cpu().numpy()


def rel(a, b):
    a, b = np.asarray(a, np.float64).ravel(), np.asarray(b, np.float64).ravel()
    assert np.all(np.isfinite(a))
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("kt,vt", PAIRS)
def test_pairs_and_tile_edges(rd4, orc, dev, kt, vt):
    import torch
    # (heads, pos0, queries): a ragged last block, exactly one row block (126, 132
    # and 128 rows), a first key block alone, many blocks (key splits), f16 queries
    for i, (nh, nkv, pos0, nq, f16) in enumerate([(24, 4, 0, 1, 0), (24, 4, 31, 21, 0), (24, 4, 33, 22, 1),
                                                  (16, 2, 63, 16, 0), (32, 8, 2000, 33, 0), (8, 8, 64, 129, 1)]):
        n = pos0 + nq
        k, v = rows_of(orc, kt, n, nkv, 10 * i + kt), rows_of(orc, vt, n, nkv, 10 * i + 5 + vt)
        q = orc.randn(nq * nh * 256, 100 + i).reshape(nq, nh, 256)
        q = q.astype(np.float16) if f16 else q
        pos = pos0 + np.arange(nq, dtype=np.int32)
        want = orc.attn_batch(q.astype(np.float32), k, v, pos, nh, nkv, 256, 1 / 16, kt, vt, threads=8)
        got, _ = run(rd4, torch, dev, q, k, v, pos0, nh, nkv, kt, vt)
        assert rel(got, want) <= REL, (kt, vt, nh, nkv, pos0, nq)


@pytest.mark.parametrize("kt,vt", [(2, 2), (4, 5), (3, 3)])
def test_no_less_precise_than_valu_kernel(rd4, orc, dev, monkeypatch, kt, vt):
    import torch
    nh, nkv, pos0, nq = 24, 4, 3000, 64
    n = pos0 + nq
    k, v = rows_of(orc, kt, n, nkv, 1), rows_of(orc, vt, n, nkv, 2)
    q, g = orc.randn(nq * nh * 256, 3).reshape(nq, nh, 256), orc.randn(nq * nh * 256, 4).reshape(nq, nh, 256)
    want = orc.attn_batch(q, k, v, pos0 + np.arange(nq, dtype=np.int32), nh, nkv, 256, 1 / 16, kt, vt, threads=8)
    gw, want = orc.sigmoid_gate(g, want)
    a, ga = run(rd4, torch, dev, q, k, v, pos0, nh, nkv, kt, vt, gate=g)
    monkeypatch.setenv("RD4_PREFILL_GENERIC", "1")
    b, gb = run(rd4, torch, dev, q, k, v, pos0, nh, nkv, kt, vt, gate=g)
    assert np.array_equal(ga, gb)
    # measured: at or below the VALU kernel; 1.5 covers a seed's noise
    assert rel(a, want) <= 1.5 * rel(b, want) + 1e-7, (rel(a, want), rel(b, want))


@pytest.mark.parametrize("kt,vt,ks,vs,qs", [(2, 2, 1e-4, 1e-4, 1e4), (2, 3, 300.0, 3e3, 1e-3), (4, 5, 1e-3, 1e-3, 1.0),
                                            (5, 4, 50.0, 1e3, 1e-2), (3, 2, 1e-2, 1.0, 1e5)])
def test_value_ranges(rd4, orc, dev, kt, vt, ks, vs, qs):
    """Caches and queries far from 1 (f16 alone would lose or overflow them)."""
    import torch
    nh, nkv, pos0, nq = 24, 4, 200, 40
    n = pos0 + nq
    k, v = rows_of(orc, kt, n, nkv, 1, ks), rows_of(orc, vt, n, nkv, 2, vs)
    q = (orc.randn(nq * nh * 256, 3) * np.float32(qs / max(1.0, ks * qs))).reshape(nq, nh, 256)
    want = orc.attn_batch(q, k, v, pos0 + np.arange(nq, dtype=np.int32), nh, nkv, 256, 1 / 16, kt, vt, threads=8)
    got, _ = run(rd4, torch, dev, q, k, v, pos0, nh, nkv, kt, vt)
    assert rel(got, want) <= REL, rel(got, want)


def test_rows_of_mixed_size_and_zeros(rd4, orc, dev):
    """V rows from 2^-10 to 2^10 side by side, zero rows, a zero query: every row
    keeps the precision of its own largest terms."""
    import torch
    nh, nkv, pos0, nq = 24, 4, 100, 30
    n = pos0 + nq
    x = orc.randn(n * nkv * 256, 8).reshape(n, nkv, 256)
    x *= np.exp2(np.arange(n) % 21 - 10).astype(np.float32)[:, None, None]
    x[::7] = 0
    k, v = rows_of(orc, 2, n, nkv, 1), orc.store_rows(2, x.ravel())
    q = orc.randn(nq * nh * 256, 3).reshape(nq, nh, 256)
    q[3] = 0
    want = orc.attn_batch(q, k, v, pos0 + np.arange(nq, dtype=np.int32), nh, nkv, 256, 1 / 16, 2, 2, threads=8)
    got, _ = run(rd4, torch, dev, q, k, v, pos0, nh, nkv, 2, 2)
    assert rel(got, want) <= REL


@pytest.mark.parametrize("which", ["k", "v"])
def test_a_row_that_is_not_finite_stays_with_its_readers(rd4, orc, dev, which):
    """One K or V block with an infinite scale at a chunk row: queries before it are
    untouched; from it on, V's block of 32 dims (K: the whole head) is not finite."""
    import torch
    nh, nkv, pos0, nq, bad, h, b = 24, 4, 40, 50, 60, 1, 3
    n = pos0 + nq
    k, v = rows_of(orc, 2, n, nkv, 1), rows_of(orc, 2, n, nkv, 2)
    q = orc.randn(nq * nh * 256, 3).reshape(nq, nh, 256)
    clean, _ = run(rd4, torch, dev, q, k, v, pos0, nh, nkv, 2, 2)
    c = (k if which == "k" else v).reshape(n, nkv, 8, 34)
    c[bad, h, b, :2] = np.frombuffer(np.float16(np.inf).tobytes(), np.uint8)
    out = torch.full(q.shape, float("nan"), dtype=torch.float32, device=dev)
    rd4.prefill(to_dev(q, torch, dev), to_dev(k, torch, dev), to_dev(v, torch, dev), out, pos0, nh, nkv, 256, 1 / 16,
                2, 2)
    got = out.cpu().numpy()
    hit = np.zeros(got.shape, bool)
    hit[bad - pos0:, 6 * h:6 * h + 6, (slice(32 * b, 32 * b + 32) if which == "v" else slice(None))] = True
    assert np.array_equal(got[~hit], clean[~hit])
    assert not np.isfinite(got[hit]).any()


def test_an_f16_v_value_that_is_not_finite_stays_with_its_readers(rd4, orc, dev):
    """The same for single values of an f16 V cache beside a quantized K: the dims
    that hold them are infinite or NaN from the key's row on, everything else as
    without them."""
    import torch
    nh, nkv, pos0, nq, h = 24, 4, 40, 50, 2
    n = pos0 + nq
    k, v = rows_of(orc, 2, n, nkv, 1), rows_of(orc, 1, n, nkv, 2)
    q = orc.randn(nq * nh * 256, 3).reshape(nq, nh, 256)
    c = v.view(np.float16).reshape(n, nkv, 256)
    for bad, d in ((47, 5), (63, 200), (64, 31), (75, 128)):
        c[bad, h, d] = 0
    clean, _ = run(rd4, torch, dev, q, k, v, pos0, nh, nkv, 2, 1)
    hit = np.zeros(clean.shape, bool)
    for bad, d, x in ((47, 5, np.inf), (63, 200, -np.inf), (64, 31, np.nan), (75, 128, np.inf)):
        c[bad, h, d] = x
        hit[bad - pos0:, 6 * h:6 * h + 6, d] = True
    out = torch.full(q.shape, float("nan"), dtype=torch.float32, device=dev)
    rd4.prefill(to_dev(q, torch, dev), to_dev(k, torch, dev), to_dev(v, torch, dev), out, pos0, nh, nkv, 256, 1 / 16,
                2, 1)
    got = out.cpu().numpy()
    assert np.array_equal(got[~hit], clean[~hit])
    assert not np.isfinite(got[hit]).any()
    assert np.all(got[7:, 6 * h:6 * h + 6, 5] == np.inf)


@pytest.mark.parametrize("vt", [1, 2, 5])
def test_q4_1_keys_no_less_precise_than_valu_kernel(rd4, orc, dev, monkeypatch, vt):
    """q4_1 K values fill both parts of their f16 pairs (d * q + m), so the product of
    the two remainders counts: without it the error over these short contexts is 1.04
    to 1.23 times the VALU kernel's, with it 0.88 to 0.96 (sums of five seeds' errors)."""
    import torch
    nh, nkv = 24, 4
    for nq, pos0 in ((1, 30), (33, 0)):
        err = {"0": 0.0, "1": 0.0}
        for seed in range(5):
            n = pos0 + nq
            k, v = rows_of(orc, 5, n, nkv, 10 * seed + 1), rows_of(orc, vt, n, nkv, 10 * seed + 2)
            q = orc.randn(nq * nh * 256, 10 * seed + 3).reshape(nq, nh, 256)
            want = orc.attn_batch(q, k, v, pos0 + np.arange(nq, dtype=np.int32), nh, nkv, 256, 1 / 16, 5, vt, threads=8)
            for env in err:
                monkeypatch.setenv("RD4_PREFILL_GENERIC", env)
                err[env] += rel(run(rd4, torch, dev, q, k, v, pos0, nh, nkv, 5, vt)[0], want)
        assert err["0"] <= err["1"], (nq, pos0, err)


@pytest.mark.parametrize("kt,vt,nh,nkv,pos0,nq,r0", [(3, 3, 24, 4, 3061, 990, 942), (2, 2, 32, 8, 2300, 855, 807),
                                                     (4, 5, 24, 4, 281, 941, 893), (3, 3, 16, 2, 0, 1660, 780)])
def test_long_sums_no_less_precise_than_valu_kernel(rd4, orc, dev, monkeypatch, kt, vt, nh, nkv, pos0, nq, r0):
    """Calls whose CTAs each sum all of a row's keys (row blocks enough for the GPU: one
    split; the last case: two, and rows that end in the first): 48 rows from r0 on. With
    O rounded at every product the error is 1.06 to 1.19 times the VALU kernel's, with one
    rounding per key block 0.51 to 0.79."""
    import torch
    n = pos0 + nq
    k, v = rows_of(orc, kt, n, nkv, 1), rows_of(orc, vt, n, nkv, 2)
    q, rows = orc.randn(nq * nh * 256, 3).reshape(nq, nh, 256), slice(r0, r0 + 48)
    pos = pos0 + np.arange(nq, dtype=np.int32)
    want = orc.attn_batch(q[rows], k, v, pos[rows], nh, nkv, 256, 1 / 16, kt, vt, threads=8)
    a = run(rd4, torch, dev, q, k, v, pos0, nh, nkv, kt, vt)[0][rows]
    monkeypatch.setenv("RD4_PREFILL_GENERIC", "1")
    b = run(rd4, torch, dev, q, k, v, pos0, nh, nkv, kt, vt)[0][rows]
    assert rel(a, want) <= rel(b, want), (rel(a, want), rel(b, want))
