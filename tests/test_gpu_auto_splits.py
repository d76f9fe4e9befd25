"""The automatic split count where the CTAs of a split do not divide the CUs (three
token pairs, three kv heads) and where they alone exceed them (one split), against
the f64 oracle."""
import numpy as np
import pytest

from gpu_util import check_close, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [1, 2])
@pytest.mark.parametrize("nh,nkv,t0,n_tok", [(24, 4, 2000, 5), (24, 4, 1500, 6), (12, 3, 3000, 1), (12, 3, 2100, 4),
                                             (24, 4, 100, 140)])
def test_tokens_at_automatic_splits(rd4, orc, dev, t, nh, nkv, t0, n_tok):
    import torch
    n, seed = t0 + n_tok, 7 * t0 + n_tok
    k, v = orc.store_rows(t, orc.randn(n * nkv * 256, seed)), orc.store_rows(t, orc.randn(n * nkv * 256, seed + 1))
    q = orc.randn(n_tok * nh * 256, seed + 2).reshape(n_tok, nh, 256)
    want = orc.attn_batch(q, k, v, t0 + np.arange(n_tok, dtype=np.int32), nh, nkv, 256, 1 / 16, t, t, threads=8)
    out = torch.full(q.shape, float("nan"), dtype=torch.float32, device=dev)
    rd4.attn_decode_tokens(to_dev(q, torch, dev), to_dev(k, torch, dev), to_dev(v, torch, dev), out, t0, n_tok, nh, nkv,
                           256, 1 / 16, t, t)
    torch.cuda.synchronize()
    check_close(out.cpu().numpy(), want, "tokens %d at %d, %d/%d" % (n_tok, t0, nh, nkv))
