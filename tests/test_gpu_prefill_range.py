"""Prefill over quantized caches where values lie far apart: blocks of one V row,
blocks of one K row, parts of one query, and values that are not finite. The path
holds its operands as f16 pairs; what such a pair cannot hold takes an f32 path, so
the results keep the tolerance of the path's other tests (3e-6, there derived), here
for each 32-dim block of the output by itself, and are infinite or NaN where the
VALU kernel's are."""
import numpy as np
import pytest

from gpu_util import to_dev

pytestmark = pytest.mark.gpu
REL = 3e-6
NH, NKV, HD = 24, 4, 256


def run(rd4, torch, dev, q, k, v, pos0, kt, vt):
    out = torch.full(q.shape, float("nan"), dtype=torch.float32, device=dev)
    rd4.prefill(to_dev(q, torch, dev), to_dev(k, torch, dev), to_dev(v, torch, dev), out, pos0, NH, NKV, HD, 1 / 16, kt, vt)
    torch.cuda.synchronize()
    return out.cpu().numpy()


def block_error(got, want):
    """Largest relative error (2-norm) of a (query, head, 32-dim block)."""
    a, b = got.astype(np.float64).reshape(-1, 32), np.asarray(want, np.float64).reshape(-1, 32)
    assert np.isfinite(a).all()
    ref = np.linalg.norm(b, axis=1)
    return float((np.linalg.norm(a - b, axis=1)[ref > 0] / ref[ref > 0]).max())


def oracle(orc, q, k, v, pos0, kt, vt):
    return orc.attn_batch(q.astype(np.float32), k, v, pos0 + np.arange(len(q), dtype=np.int32), NH, NKV, HD, 1 / 16,
                          kt, vt, threads=8)


# V: which blocks are 2^-bits of the others: block 3 of every row; all but one block
# of every 16th row; one block of the row, another in each row, the rest of the huge
# row's blocks zero; whole rows
@pytest.mark.parametrize("kt,vt", [(2, 2), (3, 3), (4, 5), (1, 2), (5, 4)])
@pytest.mark.parametrize("bits", [13, 17, 21, 25])
@pytest.mark.parametrize("how", ["block", "huge", "huge_zero", "rows"])
def test_v_blocks_far_apart(rd4, orc, dev, kt, vt, bits, how):
    import torch
    pos0, nq = 90, 40
    n, f = pos0 + nq, np.float32(2.0 ** -bits)
    x = orc.randn(n * NKV * HD, 2).reshape(n, NKV, 8, 32) * np.float32(2000)
    if how == "block":
        x[:, :, 3] *= f
    elif how == "rows":
        x[:n // 2] *= f
    else:
        small = np.ones((n, 8), bool)
        small[5::16, 2] = False
        x[small.nonzero()[0], :, small.nonzero()[1]] *= f
        if how == "huge_zero":
            for r in range(5, n, 16):
                x[r, :, np.arange(8) != 2] = 0
    k, v = orc.store_rows(kt, orc.randn(n * NKV * HD, 1)), orc.store_rows(vt, x.ravel())
    q = orc.randn(nq * NH * HD, 3).reshape(nq, NH, HD)
    err = block_error(run(rd4, torch, dev, q, k, v, pos0, kt, vt), oracle(orc, q, k, v, pos0, kt, vt))
    assert err <= REL, err


@pytest.mark.parametrize("kt,vt", [(2, 2), (3, 3), (4, 5), (5, 1)])
@pytest.mark.parametrize("bits", [15, 19, 23, 26])
@pytest.mark.parametrize("q_tiny", [False, True])
def test_k_blocks_and_queries_far_apart(rd4, orc, dev, kt, vt, bits, q_tiny):
    """K's block 5 is 2^bits of the others; the queries are zero there (the scores
    come from the small blocks alone) or 2^-bits of their other values."""
    import torch
    pos0, nq = 90, 40
    n = pos0 + nq
    x = orc.randn(n * NKV * HD, 1).reshape(n, NKV, 8, 32) * np.float32(2000 * 2.0 ** -bits)
    x[:, :, 5] *= np.float32(2.0 ** bits)
    q = orc.randn(nq * NH * HD, 3).reshape(nq, NH, 8, 32) * np.float32(2.0 ** bits / 2000)
    q[:, :, 5] *= np.float32(2.0 ** -bits if q_tiny else 0)
    q = q.reshape(nq, NH, HD)
    k, v = orc.store_rows(kt, x.ravel()), orc.store_rows(vt, orc.randn(n * NKV * HD, 2))
    err = block_error(run(rd4, torch, dev, q, k, v, pos0, kt, vt), oracle(orc, q, k, v, pos0, kt, vt))
    assert err <= REL, err


def like_valu(rd4, torch, dev, monkeypatch, q, k, v, pos0, kt, vt):
    """The call on the matrix cores and in the VALU kernel: infinite and NaN in the
    same places, and as close elsewhere as two f32 results are."""
    got = run(rd4, torch, dev, q, k, v, pos0, kt, vt)
    monkeypatch.setenv("RD4_PREFILL_GENERIC", "1")
    want = run(rd4, torch, dev, q, k, v, pos0, kt, vt)
    fin, inf = np.isfinite(want), np.isinf(want)
    assert np.argwhere(np.isfinite(got) != fin)[:5].tolist() == []
    assert np.argwhere(np.isnan(got) != np.isnan(want))[:5].tolist() == []
    assert (got[inf] == want[inf]).all()
    assert np.linalg.norm(got[fin] - want[fin]) <= 2 * REL * np.linalg.norm(want[fin])
    return want


@pytest.mark.parametrize("kt,vt", [(1, 2), (1, 5), (2, 2), (4, 5), (3, 1)])
@pytest.mark.parametrize("sign", [-1.0, 1.0])
def test_infinite_k(rd4, orc, dev, monkeypatch, kt, vt, sign):
    """K rows with an infinite value (f16) or an infinite block scale over values of
    one sign: scores of -inf leave the key out, +inf make the head NaN."""
    import torch
    pos0, nq, h = 60, 40, 2
    n = pos0 + nq
    x = orc.randn(n * NKV * HD, 1).reshape(n, NKV, HD)
    x[:, :, 64:96] = 0.5 + np.abs(x[:, :, 64:96])
    q = orc.randn(nq * NH * HD, 3).reshape(nq, NH, HD)
    q[:, :, 64:96] = 0.1 + np.abs(q[:, :, 64:96])
    k, v = orc.store_rows(kt, x.ravel()), orc.store_rows(vt, orc.randn(n * NKV * HD, 2))
    # (q4_0 / q5_0 store d < 0 with levels below the offset where the largest value is
    # positive; q4_1 as d and m)
    rows = k.view(np.uint8).reshape(n, NKV, -1)
    for r in (0, 7, 61, 64, 95):
        if kt == 1:
            rows.view(np.float16)[r, h, 70] = sign * np.inf
        else:
            b = rows[r, h].reshape(8, -1)[2]
            d = b[:2].view(np.float16)
            d[0] = np.copysign(np.inf, sign * float(d[0]))
    want = like_valu(rd4, torch, dev, monkeypatch, q, k, v, pos0, kt, vt)
    assert np.isfinite(want[:, 6 * h + 6:]).all() and (kt != 1 or np.isfinite(want).all() == (sign < 0))


@pytest.mark.parametrize("kt,vt", [(2, 2), (1, 3)])
def test_infinite_queries(rd4, orc, dev, monkeypatch, kt, vt):
    """An infinite query value (scores of -inf and +inf, or of -inf alone) and queries
    near f32's largest. A NaN query gives NaN (the VALU kernel counts a row without
    any score as one without keys: 0), and leaves the others of its CTA alone."""
    import torch
    pos0, nq = 60, 40
    n = pos0 + nq
    x = orc.randn(n * NKV * HD, 1).reshape(n, NKV, HD)
    x[:, 1, 9] = 0.3 + np.abs(x[:, 1, 9])  # dim 9 of kv head 1: above 0 in every key
    k, v = orc.store_rows(kt, x.ravel()), orc.store_rows(vt, orc.randn(n * NKV * HD, 2))
    q = orc.randn(nq * NH * HD, 3).reshape(nq, NH, HD)
    q[3, 2, 40], q[9, 7, 9], q[17, 8, 9] = np.inf, -np.inf, np.inf
    q[25] *= np.float32(2.0 ** 120)  # finite: one key has all the weight
    like_valu(rd4, torch, dev, monkeypatch, q, k, v, pos0, kt, vt)
    monkeypatch.delenv("RD4_PREFILL_GENERIC")
    clean = run(rd4, torch, dev, q, k, v, pos0, kt, vt)
    q[30, 20, 0] = np.nan
    got = run(rd4, torch, dev, q, k, v, pos0, kt, vt)
    assert np.isnan(got[30, 20]).all()
    clean[30, 20] = got[30, 20]
    assert np.array_equal(got, clean, equal_nan=True)


@pytest.mark.parametrize("kt,vt", [(2, 2), (3, 3), (1, 5), (5, 4), (2, 1)])
def test_v_that_is_not_finite(rd4, orc, dev, monkeypatch, kt, vt):
    """Infinite and NaN V values, a single one of f16, a block scale (or q4_1's
    offset) of the quantized types."""
    import torch
    pos0, nq, h = 60, 40, 3
    n = pos0 + nq
    k, v = orc.store_rows(kt, orc.randn(n * NKV * HD, 1)), orc.store_rows(vt, orc.randn(n * NKV * HD, 2))
    q = orc.randn(nq * NH * HD, 3).reshape(nq, NH, HD)
    rows = v.view(np.uint8).reshape(n, NKV, -1)
    for r, b, val in ((1, 0, np.inf), (63, 2, -np.inf), (64, 3, np.nan), (97, 7, np.inf)):
        if vt == 1:
            rows.view(np.float16)[r, h, 32 * b + r % 32] = val
        else:
            rows[r, h].reshape(8, -1)[b][2 * (vt == 5):][:2].view(np.float16)[0] = val
    like_valu(rd4, torch, dev, monkeypatch, q, k, v, pos0, kt, vt)
