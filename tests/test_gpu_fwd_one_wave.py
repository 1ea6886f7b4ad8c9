"""Forwards of short key ranges on one wave per 32 queries (FMHA_FWD_FEW=1, and by rule): blocks that end within 32 or 64 keys, heads of a
few rows, rows that end before the kernel's width, run-time row layouts, and the lines of the rule."""
import numpy as np
import pytest
import torch

import oracle
from nvfuserexamples_amd import capi
from conftest import make_qkv, pad_mask, f32

pytestmark = pytest.mark.gpu

TDT = {"fp16": torch.float16, "bf16": torch.bfloat16}
BAR = {"fp16": (2e-3, 2.0 ** -11), "bf16": (2e-2, 2.0 ** -8)}   # as in the other forward tests: |O - oracle|, LSE beside 1e-3


@pytest.mark.parametrize("packed", [False, True], ids=["", "packed"])
@pytest.mark.parametrize("bh,sq,sk,d,dtype,causal,p,mask", [
    (6, 16, 16, 32, "fp16", False, 0.0, None), (6, 33, 65, 24, "fp16", False, 0.1, "pad"), (6, 63, 63, 48, "bf16", True, 0.0, None),
    (6, 64, 64, 64, "fp16", True, 0.1, None), (6, 31, 31, 96, "fp16", False, 0.1, "pad"), (6, 97, 96, 80, "fp16", False, 0.0, "len"),
    (6, 160, 160, 128, "bf16", True, 0.0, None), (6, 17, 129, 128, "fp16", False, 0.1, "len"), (6, 1, 40, 256, "fp16", False, 0.0, "pad"),
    (6, 70, 64, 200, "fp16", True, 0.1, None), (600, 20, 20, 256, "fp16", False, 0.0, None),
])
def test_short_ranges(bh, sq, sk, d, dtype, causal, p, mask, packed):
    q, k, v = make_qkv(bh, sq, sk, d, seed=sk + d, dtype=dtype)
    kw, okw = dict(causal=causal), dict(causal=causal)
    if mask:
        m = pad_mask(2, sk, sk // 2, sk).to(TDT[dtype])
        lens = (m[:, 0, 0] == 0).sum(-1).to(torch.int32)
        if mask == "pad":
            kw["mask"] = m.cuda()
        else:
            kw["kv_len"] = lens.cuda()
        okw["mask"] = f32(m) if mask == "pad" else np.where(np.arange(sk)[None, None, None] < lens.numpy()[:, None, None, None], 0.0, -np.inf).astype(np.float32)
    if p:
        kw.update(drop_kind=capi.DROP_PHILOX, p_drop=p, seed=9, offset=4)
        okw.update(philox=True, p_drop=p, seed=9, offset=4)
    ins = [t.cuda() for t in (q, k, v)]
    if packed:
        ins = [t.view(2, bh // 2, t.shape[1], d).transpose(1, 2).contiguous().transpose(1, 2) for t in ins]
    o, lse, _, _ = capi.fwd(*ins, want_lse=True, scale=d ** -0.5, **kw)
    ref = oracle.attention(f32(q), f32(k), f32(v), want=("o", "lse"), **okw)
    bar, unit = BAR[dtype]
    assert np.abs(f32(o.cpu()).reshape(ref["o"].shape) - ref["o"]).max() <= bar * max(1.0, np.abs(ref["o"]).max() / 2)
    lse = lse.cpu().numpy().reshape(ref["lse"].shape)
    assert np.abs(lse - ref["lse"]).max() <= 1e-3 + unit * np.abs(ref["lse"]).max()


@pytest.mark.parametrize("d,sk,causal,here", [
    (32, 64, False, True), (32, 65, False, False), (32, 96, True, True), (32, 97, True, False), (64, 64, False, False), (64, 64, True, True),
    (64, 65, True, False), (96, 96, False, True), (96, 97, False, False), (128, 128, False, False), (128, 129, False, True), (128, 161, False, False),
    (256, 64, True, True), (256, 65, True, False),
])
def test_where_the_rule_lies(d, sk, causal, here, monkeypatch):
    """It looks at a head's shape only: a head's bits do not depend on how many others there are."""
    monkeypatch.delenv("FMHA_FWD_FEW", raising=False)
    ins = [t.cuda() for t in make_qkv(3, sk, sk, d, seed=d)]
    got = capi.fwd(*ins, causal=causal, want_lse=True)
    many = capi.fwd(*[t.repeat(300, 1, 1) for t in ins], causal=causal, want_lse=True)
    monkeypatch.setenv("FMHA_FWD_FEW", "1" if here else "0")
    want = capi.fwd(*ins, causal=causal, want_lse=True)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    if here:
        assert torch.equal(many[0][:3], got[0]) and torch.equal(many[0][-3:], got[0])
