"""The fused epilogue over chunks long enough that a wave takes several rows of a
token (fewer CTAs per token as the chunk grows): every output byte equals the
unfused launches', at row counts that leave waves of the last group idle."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kt,vt,hd,nh,nkv,n_rot,n_tok", [
    (2, 2, 256, 24, 4, 64, 700),    # 6 CTAs per token: a second row for some waves
    (4, 5, 256, 24, 4, 64, 2100),   # 2 per token
    (1, 3, 256, 6, 1, 256, 4200),   # 1 per token, 8 rows over 4 waves, every pair rotated
    (2, 1, 256, 7, 7, 64, 4100),    # 21 rows
    (2, 2, 512, 3, 3, 512, 4100),   # two 256-element groups per row, 256 angles
    (2, 2, 64, 9, 3, 0, 4100),      # 16 lanes of a wave, no rotation
])
def test_long_chunks_equal_unfused(rd4, dev, kt, vt, hd, nh, nkv, n_rot, n_tok):
    import torch
    g = torch.Generator(device="cuda").manual_seed(hd + n_tok)
    qg = torch.randn(n_tok, nh, 2, hd, generator=g, device=dev)
    k, v = (torch.randn(n_tok, nkv, hd, generator=g, device=dev) for _ in range(2))
    qw, kw = (1 + 0.1 * torch.randn(hd, generator=g, device=dev) for _ in range(2))
    pos = torch.arange(5, 5 + n_tok, dtype=torch.int32, device=dev)
    krb, vrb = rd4.kv_row_bytes(kt, hd), rd4.kv_row_bytes(vt, hd)
    caches = [torch.full(((n_tok + 9) * nkv * rb,), 77, dtype=torch.uint8, device=dev) for rb in (krb, vrb, krb, vrb)]
    q1, g1, k1 = torch.empty(n_tok, nh, hd, device=dev), torch.empty(n_tok, nh, hd, device=dev), torch.empty_like(k)
    rd4.qk_norm_rope_append(qg, k, v, qw, kw, 1e-6, n_rot, 1e7, pos, n_tok, nh, nkv, hd, q1, caches[0], caches[1], kt, vt,
                            gate_out=g1, k_out=k1)
    q2, k2 = qg[:, :, 0].contiguous(), k.clone()
    rd4.rms_norm(q2, qw, q2, n_tok * nh, hd, 1e-6)
    rd4.rms_norm(k2, kw, k2, n_tok * nkv, hd, 1e-6)
    if n_rot:
        rd4.rope(q2, n_tok, nh, hd, n_rot, 1e7, pos)
        rd4.rope(k2, n_tok, nkv, hd, n_rot, 1e7, pos)
    w = n_tok * nkv * hd
    rd4.kv_store_rows(kt, k2, caches[2][5 * nkv * krb:], w)
    rd4.kv_store_rows(vt, v, caches[3][5 * nkv * vrb:], w)
    torch.cuda.synchronize()
    for a, b in ((q1, q2), (g1, qg[:, :, 1].contiguous()), (k1, k2)):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))
    assert torch.equal(caches[0], caches[2]) and torch.equal(caches[1], caches[3])
