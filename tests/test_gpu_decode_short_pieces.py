"""Decode steps of few heads: pieces of the key range below 1024 keys (128 keys and more, by a model of the step's time), ranges of 513 keys and more,
the merge of up to 64 pieces, a workspace that only has room for the longer pieces, and steps that the model keeps whole."""
import ctypes as C
import numpy as np
import pytest
import torch

import oracle
from nvfuserexamples_amd import capi
from conftest import make_qkv, f32

pytestmark = pytest.mark.gpu

O_TOL = {"fp16": 2e-3, "bf16": 2e-2}       # as in test_gpu_decode.py


def _need(bh, sq, sk, d):
    P = capi.FwdParams()
    P.bh, P.sq, P.sk, P.d = bh, sq, sk, d
    P.scale = d ** -0.5
    capi._sync_env()
    return capi.lib().fmha_fwd_workspace_bytes(C.byref(P))


@pytest.mark.parametrize("bh,sq,sk,d,dtype", [
    (3, 4, 513, 128, "fp16"), (2, 3, 2047, 128, "bf16"), (2, 1, 1701, 128, "fp16"), (3, 2, 2049, 64, "fp16"), (1, 4, 8321, 128, "fp16"),
    (12, 1, 1939, 128, "fp16"), (40, 1, 3980, 64, "bf16"), (2, 2, 9000, 128, "fp16"),
])
def test_short_pieces(bh, sq, sk, d, dtype):
    assert _need(bh, sq, sk, d) > 0
    q, k, v = make_qkv(bh, sq, sk, d, seed=sk, dtype=dtype)
    lens = torch.tensor([1 + (sk - 1) * (i + 1) // bh for i in range(bh)], dtype=torch.int32)   # the first head's last pieces are empty
    qc, kc, vc = q.cuda(), k.cuda(), v.cuda()
    o, lse, _, _ = capi.fwd(qc, kc, vc, kv_len=lens.cuda(), want_lse=True)
    o0, lse0, _, _ = capi.fwd(qc, kc, vc, kv_len=lens.cuda(), want_lse=True, workspace=False)
    m = np.where(np.arange(sk)[None, None] < lens.numpy()[:, None, None], 0.0, -np.inf).astype(np.float32) * np.ones((1, sq, 1), np.float32)
    ref = oracle.attention(f32(q), f32(k), f32(v), mask=m, want=("o", "lse"))
    assert np.abs(f32(o.cpu()) - ref["o"]).max() <= O_TOL[dtype]
    assert np.abs(lse.cpu().numpy() - ref["lse"]).max() <= 2e-3
    assert (lse - lse0).abs().max().item() <= 5e-4


def test_a_workspace_for_the_longer_pieces_only():
    """3 heads of four rows by 4096 keys take 32 pieces of 128; in a workspace for four of 1024 they take those."""
    bh, sq, sk, d = 3, 4, 4096, 128
    need = _need(bh, sq, sk, d)
    coarse = 4 * bh * (sq * d * 4 + sq * 4) + 512
    assert need > coarse
    q, k, v = (t.cuda() for t in make_qkv(bh, sq, sk, d, seed=1))
    o = capi.fwd(q, k, v)[0]
    ws = torch.zeros(coarse, dtype=torch.uint8, device="cuda")
    o1 = capi.fwd(q, k, v, workspace=ws)[0]
    assert ws.any()                                    # (in pieces)
    assert (o.float() - o1.float()).abs().max().item() <= 1e-3


def test_ranges_that_stay_whole():
    """.. where the model of the two times has the merge cost more than the pieces save."""
    assert _need(8, 1, 789, 64) == 0 and _need(16, 1, 700, 128) == 0 and _need(178, 1, 1660, 128) == 0 and _need(255, 4, 1500, 128) == 0
