"""The forward whose waves share 32 queries and take their blocks of keys in turn (FMHA_FWD_FEW=4|8): waves without a block, blocks
that the end of the keys, the diagonal or a mask passes through, rows whose keys are all hidden from some waves, dropout, row
layouts and head dims between the built ones, against the oracle; key counts against the mask that hides the same keys, to
the bit; and the calls that the operators' flag sends there."""
import numpy as np
import pytest
import torch

import oracle
from nvfuserexamples_amd import capi, load_ops
from conftest import f32, make_qkv

pytestmark = pytest.mark.gpu

BAR = {"fp16": (2e-3, 2.0 ** -11), "bf16": (2e-2, 2.0 ** -8)}   # as in the other forward tests: |O - oracle|, LSE beside 1e-3


@pytest.fixture(params=["4", "8"])
def waves(request, monkeypatch):
    monkeypatch.setenv("FMHA_FWD_FEW", request.param)
    return int(request.param)


def _check(o, lse, ref, dtype):
    bar, unit = BAR[dtype]
    got = f32(o.float().cpu()).reshape(ref["o"].shape)
    assert np.abs(got - ref["o"]).max() <= bar * max(1.0, np.abs(ref["o"]).max() / 2)
    l, want = lse.float().cpu().numpy().reshape(ref["lse"].shape), ref["lse"]
    assert np.array_equal(np.isneginf(l), np.isneginf(want))
    live = np.isfinite(want)
    assert np.abs(l[live] - want[live]).max(initial=0.0) <= 5e-3 + unit * np.abs(want[live]).max(initial=0.0)


@pytest.mark.parametrize("sq,sk,d,dtype,causal,p", [
    (1, 1, 64, "fp16", False, 0.0), (5, 63, 64, "bf16", False, 0.0), (33, 65, 64, "fp16", True, 0.0), (32, 256, 64, "fp16", False, 0.1),
    (100, 300, 32, "fp16", False, 0.0), (130, 130, 64, "bf16", True, 0.1), (257, 700, 64, "fp16", False, 0.0), (300, 90, 64, "fp16", True, 0.0),
    (31, 33, 128, "fp16", False, 0.0), (64, 129, 128, "bf16", True, 0.0), (200, 270, 96, "fp16", False, 0.1), (7, 545, 80, "bf16", False, 0.0),
    (65, 31, 256, "fp16", False, 0.0), (40, 161, 256, "bf16", True, 0.1), (33, 200, 200, "fp16", True, 0.0), (12, 40, 8, "fp16", False, 0.0),
])
def test_shared_queries_match_the_oracle(sq, sk, d, dtype, causal, p, waves):
    bh = 3
    q, k, v = make_qkv(bh, sq, sk, d, seed=sq + sk, std=1.0 if d <= 64 else 0.5, dtype=dtype)
    kw = dict(drop_kind=capi.DROP_PHILOX, p_drop=p, seed=11, offset=2) if p else {}
    o, lse, _, _ = capi.fwd(q.cuda(), k.cuda(), v.cuda(), causal=causal, want_lse=True, **kw)
    okw = dict(philox=True, p_drop=p, seed=11, offset=2) if p else {}
    _check(o, lse, oracle.attention(f32(q), f32(k), f32(v), causal=causal, want=("o", "lse"), **okw), dtype)


@pytest.mark.parametrize("d,sk", [(64, 300), (128, 270), (256, 140)])
@pytest.mark.parametrize("packed", [False, True])
def test_masks_counts_and_layouts(d, sk, packed, waves, monkeypatch):
    """Live keys in one wave's blocks only, at the start or the end, none at all; the hard-masked tail left out or visited; rows
    read in place from a packed projection: the folded build's bits."""
    spans = [(0, 1), (0, 64), (64, 65), (100, 130), (sk - 1, sk), (0, sk // 2), (0, sk), (0, 0)]
    b, h = len(spans), 2
    x = torch.randn(b, sk, 3, h, d, generator=torch.Generator().manual_seed(sk)).half() * (0.5 if d > 64 else 1.0)
    q, k, v = (x[:, :, i].transpose(1, 2) for i in range(3))
    fold = [t.reshape(b * h, sk, d).contiguous() for t in (q, k, v)]
    for hidden in (-10000.0, float("-inf")):
        m = torch.full((b, 1, 1, sk), hidden)
        for i, (lo, hi) in enumerate(spans):
            m[i, :, :, lo:hi] = 0.0
        m = m.half()
        ins = [t.cuda() for t in fold]
        o, lse, _, _ = capi.fwd(*ins, mask=m.cuda(), want_lse=True)
        if packed:
            xp = x.cuda()
            op, lp, _, _ = capi.fwd(*(xp[:, :, i].transpose(1, 2) for i in range(3)), mask=m.cuda(), want_lse=True)
            assert torch.equal(op.reshape(o.shape), o) and torch.equal(lp.reshape(lse.shape), lse)
            continue
        full = np.broadcast_to(f32(m).reshape(b, 1, 1, sk), (b, h, sk, sk)).reshape(b * h, sk, sk).copy()
        n = b * h if hidden > float("-inf") else (b - 1) * h  # (the last sequence sees nothing: zeros and -inf, below)
        _check(o[:n], lse[:n], oracle.attention(*(f32(t[:n]) for t in fold), mask=full[:n], want=("o", "lse")), "fp16")
        if n < b * h:
            assert not o[n:].any() and bool(torch.isneginf(lse[n:]).all())
        monkeypatch.setenv("FMHA_MASK_TRIM", "0")
        o2, lse2, _, _ = capi.fwd(*ins, mask=m.cuda(), want_lse=True)
        monkeypatch.delenv("FMHA_MASK_TRIM")
        assert torch.equal(o, o2) and torch.equal(lse, lse2)
    lens = torch.tensor([1, 31, 32, 33, sk - 1, sk, 64, 65], dtype=torch.int32)
    m = torch.where(torch.arange(sk)[None] < lens[:, None], 0.0, -10000.0).view(b, 1, 1, sk).half().cuda()
    for causal in (False, True):
        a = capi.fwd(*ins, mask=m, causal=causal, want_lse=True)
        c = capi.fwd(*ins, kv_len=lens.cuda(), causal=causal, want_lse=True)
        assert torch.equal(a[0], c[0]) and torch.equal(a[1], c[1])


@pytest.mark.parametrize("bh,sq,sk,d,causal", [(2, 200, 200, 128, False), (8, 600, 600, 64, True), (4, 96, 5000, 64, False), (17, 1000, 1000, 128, False), (3, 200, 300, 256, True)])
def test_the_flag_decides(bh, sq, sk, d, causal, monkeypatch):
    """Without FMHA_FLAG_SPLIT_KEYS a launch of few workgroups does not take this kernel: at these shapes, where the other kernels have no line in the
    number of heads, a head's bits are those it has among twelve times as many.  The operator, which sets the flag, takes this kernel where
    the rule does and agrees with the other kernels to the rounding of O.  (4 x 96 x 5000 stays in pieces, 17 x 1000 is too large.)"""
    monkeypatch.delenv("FMHA_FWD_FEW", raising=False)
    q, k, v = (t.cuda() for t in make_qkv(bh, sq, sk, d, seed=d, std=0.5))
    plain = capi.fwd(q, k, v, causal=causal, want_lse=True, workspace=False)
    many = capi.fwd(*(t.repeat(12, 1, 1) for t in (q, k, v)), causal=causal, want_lse=True, workspace=False)
    assert torch.equal(many[0][-bh:], plain[0]) and torch.equal(many[1][-bh:], plain[1])
    flagged = capi.fwd(q, k, v, causal=causal, want_lse=True, flags=4)
    ops = load_ops()
    got = ops.fmha_fwd(q, k, v, None, 0.0, causal, 0.0, 0, 0, None)
    assert torch.equal(got[0], flagged[0]) and torch.equal(got[1], flagged[1])
    assert (flagged[0].float() - plain[0].float()).abs().max() <= 2e-3 and (flagged[1] - plain[1]).abs().max() <= 2e-3
    monkeypatch.setenv("FMHA_FWD_FEW", "8" if d != 256 and sk > 768 and bh * ((sq + 31) // 32) <= 256 else "4")
    few = capi.fwd(q, k, v, causal=causal, want_lse=True)
    here = (bh, sq, sk, d) not in ((4, 96, 5000, 64), (17, 1000, 1000, 128))
    assert torch.equal(few[0], flagged[0]) == here
