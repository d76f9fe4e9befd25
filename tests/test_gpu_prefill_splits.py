"""Prefill calls whose row blocks leave CUs idle run in key splits that a merge
launch folds: few queries over many keys (up to the 64 splits a wave of the merge
holds), row-block counts that are no multiple of 8, splits that hold no key of the
early rows, and a gate, against the f64 oracle. The f16 path rounds queries and
probabilities to f16 (the attention tolerance); the quantized path computes in 32
bits (its tests' tolerance)."""
import numpy as np
import pytest

from gpu_util import check_close, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [1, 2])
@pytest.mark.parametrize("nh,nkv,pos0,nq", [(24, 4, 4100, 1), (24, 4, 4095, 16), (24, 4, 2000, 23), (32, 8, 777, 57),
                                            (16, 2, 300, 97), (6, 1, 0, 300), (12, 3, 63, 201), (24, 4, 0, 400)])
def test_split_calls_match_oracle(rd4, orc, dev, t, nh, nkv, pos0, nq):
    import torch
    n, seed = pos0 + nq, 13 * pos0 + nq
    k, v = orc.store_rows(t, orc.randn(n * nkv * 256, seed)), orc.store_rows(t, orc.randn(n * nkv * 256, seed + 1))
    q, g = orc.randn(nq * nh * 256, seed + 2).reshape(nq, nh, 256), orc.randn(nq * nh * 256, seed + 3).reshape(nq, nh, 256)
    rows = np.unique(np.linspace(0, nq - 1, 40).astype(np.int32))
    want = orc.attn_batch(q[rows], k, v, pos0 + rows, nh, nkv, 256, 1 / 16, t, t, threads=8)
    _, want = orc.sigmoid_gate(g[rows], want)
    out = torch.full(q.shape, float("nan"), dtype=torch.float32, device=dev)
    rd4.prefill(to_dev(q, torch, dev), to_dev(k, torch, dev), to_dev(v, torch, dev), out, pos0, nh, nkv, 256, 1 / 16, t, t,
                gate=to_dev(g, torch, dev))
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert np.all(np.isfinite(got))
    check_close(got[rows].ravel(), np.asarray(want).ravel(), "prefill %d/%d pos0 %d n %d" % (nh, nkv, pos0, nq))
    if t != 1:
        want = np.asarray(want, np.float64).reshape(got[rows].shape)
        assert np.linalg.norm(got[rows] - want) <= 3e-6 * np.linalg.norm(want)


@pytest.mark.parametrize("kt,vt", [(1, 1), (2, 2), (4, 5), (1, 2), (3, 1)])
def test_a_split_whose_scores_are_all_nan_stays_nan(rd4, orc, dev, kt, vt):
    """One K row that is NaN at the first key of a split (8 f16 or 15 quantized
    one-block splits): the query at that position attends no other key of its
    split, so the split's running max never leaves -inf. From the row on the head
    is NaN, before it and in the other heads nothing changes."""
    import torch
    nh, nkv, pos0, nq, h = 24, 4, 400, 60, 1
    n = pos0 + nq
    k, v = orc.store_rows(kt, orc.randn(n * nkv * 256, 1)), orc.store_rows(vt, orc.randn(n * nkv * 256, 2))
    q = to_dev(orc.randn(nq * nh * 256, 3).reshape(nq, nh, 256), torch, dev)

    def run(kb):
        out = torch.zeros(q.shape, dtype=torch.float32, device=dev)
        rd4.prefill(q, to_dev(kb, torch, dev), to_dev(v, torch, dev), out, pos0, nh, nkv, 256, 1 / 16, kt, vt)
        torch.cuda.synchronize()
        return out.cpu().numpy()

    clean = run(k)
    for bad in (416, 447, 448):  # 448 starts a block of 32 and of 64 keys, 416 one of 32
        kb = k.copy()
        kb.view(np.uint8).reshape(n, nkv, -1)[bad, h, :2] = np.frombuffer(np.float16(np.nan).tobytes(), np.uint8)
        got, hit = run(kb), np.zeros(clean.shape, bool)
        hit[bad - pos0:, 6 * h:6 * h + 6] = True
        assert np.isnan(got[hit]).all(), bad
        assert np.array_equal(got[~hit], clean[~hit]), bad


@pytest.mark.parametrize("kt,vt", [(1, 1), (2, 2), (4, 5), (1, 2), (3, 1)])
def test_a_split_whose_scores_are_all_minus_infinity_keeps_its_v(rd4, orc, dev, kt, vt):
    """One key whose scores are -inf and whose V is infinite, the first of a split: the
    query at its position attends no other key of the split. Its weight is 0, and
    0 * inf is NaN in V's dims, as where the key stands inside a split; the other dims
    are those of the key left out."""
    import torch
    nh, nkv, pos0, nq, h, b = 24, 4, 400, 60, 1, 2
    n = pos0 + nq
    x = orc.randn(n * nkv * 256, 1).reshape(n, nkv, 256)
    x[:, :, 64:96] = 0.5 + np.abs(x[:, :, 64:96])
    q = orc.randn(nq * nh * 256, 3).reshape(nq, nh, 256)
    q[:, :, 64:96] = 0.1 + np.abs(q[:, :, 64:96])
    k, v = orc.store_rows(kt, x.ravel()), orc.store_rows(vt, orc.randn(n * nkv * 256, 2))
    q = to_dev(q, torch, dev)

    def run(kb, vb):
        out = torch.zeros(q.shape, dtype=torch.float32, device=dev)
        rd4.prefill(q, to_dev(kb, torch, dev), to_dev(vb, torch, dev), out, pos0, nh, nkv, 256, 1 / 16, kt, vt)
        torch.cuda.synchronize()
        return out.cpu().numpy()

    for bad in (447, 448):  # inside a split; the first key of one (of 32 and of 64 keys)
        kb, vb = k.copy(), v.copy()
        krow = kb.view(np.uint8).reshape(n, nkv, -1)[bad, h]
        d = krow.view(np.float16)[70:71] if kt == 1 else krow.reshape(8, -1)[b, :2].view(np.float16)
        d[0] = -np.inf if kt == 1 else np.copysign(np.inf, -float(d[0]))
        left_out = run(kb, v)
        vrow = vb.view(np.uint8).reshape(n, nkv, -1)[bad, h].reshape(8, -1)[b]
        vrow[:2].view(np.float16)[0] = np.inf
        got, dims = run(kb, vb)[bad - pos0, 6 * h:6 * h + 6], slice(32 * b, 32 * b + (1 if vt == 1 else 32))
        want = left_out[bad - pos0, 6 * h:6 * h + 6]
        assert np.isfinite(want).all(), bad
        assert np.isnan(got[:, dims]).all(), bad
        want[:, dims] = got[:, dims]
        assert np.array_equal(got, want, equal_nan=True), bad
