"""Prefill calls captured on streams that were given no scratch: they take none of
the scratch that a decode captured later needs, and a prefill captured with records
gives the eager call's bits on every replay."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

# (its own process: the spare scratch that rd4_init makes is handed out once)
CODE = r'''
import sys
sys.path.insert(0, "tests")
import conftest, torch
rd4 = conftest.load_package()
sys.path.insert(0, "oracle")
import oracle as orc
kt, vt, nq = int(sys.argv[1]), int(sys.argv[2]), int(sys.argv[3])
nh, nkv, hd, pos0 = 24, 4, 256, 1000
n, dev = pos0 + nq, torch.device("cuda:0")
d = lambda a: torch.from_numpy(a).to(dev)
k, v = d(orc.store_rows(kt, orc.randn(n * nkv * hd, 1))), d(orc.store_rows(vt, orc.randn(n * nkv * hd, 2)))
q = d(orc.randn(nq * nh * hd, 3).reshape(nq, nh, hd))
out, out1 = torch.empty_like(q), torch.empty(nh * hd, device=dev)
q1 = q[0].reshape(-1).clone()
pre = lambda: rd4.prefill(q, k, v, out, pos0, nh, nkv, hd, 1 / 16, kt, vt)
dec = lambda: rd4.attn_decode(q1, k, v, out1, n - 1, nh, nkv, hd, 1 / 16, kt, vt)
pre()
dec()
torch.cuda.synchronize()
want, want1 = out.clone(), out1.clone()
assert rd4.lib().rd4_init() == 0
s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
g1, g2 = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
with torch.cuda.graph(g1, stream=s1):
    pre()
with torch.cuda.graph(g2, stream=s2):
    dec()
for i in range(3):
    out.fill_(float("nan"))
    out1.fill_(float("nan"))
    torch.cuda.synchronize()
    g1.replay()
    g2.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, want), "prefill, replay %d" % i
    assert torch.equal(out1, want1), "decode, replay %d" % i
    pre()  # eager work between the replays
    torch.cuda.synchronize()
print("ok")
'''


@pytest.mark.parametrize("kt,vt,nq", [(2, 2, 64), (4, 5, 33), (1, 1, 201), (1, 1, 512)])
def test_prefill_then_decode_captured_on_new_streams(kt, vt, nq):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", CODE, str(kt), str(vt), str(nq)], cwd=root, capture_output=True, text=True,
                       timeout=180)
    assert r.returncode == 0 and "ok" in r.stdout, r.stdout + r.stderr
