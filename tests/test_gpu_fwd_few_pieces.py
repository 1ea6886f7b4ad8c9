"""The kernel whose waves share 32 queries on pieces of the key range, and both merges of its fp32 pieces: last pieces of one key, pieces without any
visible key, row ends inside a 32-query group, head dims with and without padding, masks and key counts of the whole range, packed rows."""
import numpy as np
import pytest
import torch

import oracle
from nvfuserexamples_amd import capi
from conftest import make_qkv, f32

pytestmark = pytest.mark.gpu

SPLIT_KEYS = 4                             # FMHA_FLAG_SPLIT_KEYS
O_TOL = {"fp16": 2e-3, "bf16": 2e-2}       # as in test_gpu_decode.py


def _run(monkeypatch, pieces, *args, **kw):
    monkeypatch.setenv("FMHA_FWD_SPLIT", str(pieces))
    r = capi.fwd(*args, want_lse=True, flags=SPLIT_KEYS, **kw)
    monkeypatch.delenv("FMHA_FWD_SPLIT")
    return r[0], r[1]


@pytest.mark.parametrize("d,dtype", [(32, "fp16"), (64, "bf16"), (80, "fp16"), (96, "bf16"), (128, "fp16"), (200, "fp16"), (256, "bf16")])
@pytest.mark.parametrize("bh,sq,sk,pieces", [(2, 5, 129, 2), (3, 33, 300, 3), (4, 300, 641, 5), (2, 64, 5000, 40)])
def test_pieces_of_32_queries(bh, sq, sk, pieces, d, dtype, monkeypatch):
    q, k, v = make_qkv(bh, sq, sk, d, seed=sk, dtype=dtype)
    qc, kc, vc = q.cuda(), k.cuda(), v.cuda()
    lens = torch.tensor([sk * i // (bh - 1) for i in range(bh)], dtype=torch.int32)        # none to all
    m = torch.zeros(bh, 1, sk)
    m[:, :, sk // 3:] = -10000.0                                                           # hard-masked to the end
    m[0, :, : sk // 2] = float("-inf")
    for mask, kl in ((None, None), (m.to(q.dtype), None), (None, lens), (m.to(q.dtype), lens)):
        kw = dict(mask=None if mask is None else mask.cuda(), kv_len=None if kl is None else kl.cuda())
        o, lse = _run(monkeypatch, pieces, qc, kc, vc, **kw)
        o0, lse0 = _run(monkeypatch, 0, qc, kc, vc, **kw)
        full = np.zeros((bh, 1, sk), np.float32) if mask is None else f32(mask).copy()
        if kl is not None:
            full = np.where(np.arange(sk)[None, None] < kl.numpy()[:, None, None], full, -np.inf).astype(np.float32)
        full = np.broadcast_to(full, (bh, sq, sk)).copy()
        ref = oracle.attention(f32(q), f32(k), f32(v), mask=full, want=("o", "lse"))
        none = np.isneginf(full).all(-1)
        got, l = f32(o.cpu()), lse.cpu().numpy()
        assert (got[none] == 0).all() and np.isneginf(l[none]).all()
        assert np.abs(got[~none] - ref["o"][~none]).max() <= O_TOL[dtype]
        # (a row whose keys are all hard-masked: scores near -10 000 in fp32 and an fp32 sum of logarithms, 2^-11 each)
        assert np.abs(l[~none] - ref["lse"][~none]).max() <= 2e-3 + (2.0 ** -9 if mask is not None else 0.0)
        # fp32 pieces: the mean error is the whole launch's (both are the rounding of P and of O); a 16-bit rounding of the pieces would add to it
        e, e0 = [float(np.sqrt(np.mean((f32(x.cpu())[~none] - ref["o"][~none]) ** 2))) for x in (o, o0)]
        assert e <= 1.2 * e0 + 2e-6


@pytest.mark.parametrize("sq", [40, 600])
def test_packed_rows(sq, monkeypatch):
    b, h, sk, d = 2, 3, 700, 64
    q = make_qkv(1, b * sq, 8, h * d, seed=1)[0].reshape(b, sq, h, d).cuda()
    kv = make_qkv(1, b * sk, 8, 2 * h * d, seed=2)[0].reshape(b, sk, 2, h, d).cuda()
    args = q.transpose(1, 2), kv[:, :, 0].transpose(1, 2), kv[:, :, 1].transpose(1, 2)
    o, lse = _run(monkeypatch, 4, *args)
    o1, lse1 = _run(monkeypatch, 4, *(t.reshape(b * h, -1, d).contiguous() for t in args))
    assert torch.equal(o.reshape(b * h, sq, d), o1) and torch.equal(lse.reshape(b * h, sq), lse1)


def test_which_launches():
    """Few heads against long ranges go in pieces (fp32 where 32-query groups are taken); full launches, causal ones and callers that keep the keys together don't."""
    def need(bh, sq, sk, d, flags=SPLIT_KEYS, causal=0):
        import ctypes as C
        P = capi.FwdParams()
        P.bh, P.sq, P.sk, P.d, P.flags, P.causal, P.scale = bh, sq, sk, d, flags, causal, d ** -0.5
        capi._sync_env()
        return capi.lib().fmha_fwd_workspace_bytes(C.byref(P))
    assert need(17, 19, 1698, 256) > 0 and need(4, 256, 32768, 128) > 0 and need(1, 12, 1568, 80) > 0
    assert need(17, 19, 1698, 256, flags=0) == 0 and need(17, 19, 1698, 256, causal=1) == 0
    assert need(512, 512, 512, 64) == 0 and need(4, 100, 300, 64) == 0 and need(256, 64, 1024, 128) == 0
