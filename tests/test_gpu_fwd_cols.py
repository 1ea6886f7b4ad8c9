"""Forwards under full mask tensors with a workgroup per 32 queries and a wave per 64 keys (FMHA_FWD_COLS=1): one wave to as many as fit,
waves with one key, rows off 16-byte boundaries, rows without a visible key, and the rule that takes few workgroups there."""
import numpy as np
import pytest
import torch

import oracle
from nvfuserexamples_amd import capi, load_ops
from conftest import make_qkv, f32

pytestmark = pytest.mark.gpu

TDT = {"fp16": torch.float16, "bf16": torch.bfloat16}
BAR = {"fp16": (2e-3, 2.0 ** -11), "bf16": (2e-2, 2.0 ** -8)}   # as in the other forward tests: |O - oracle|, LSE beside 1e-3


def _check(got, want, bar):
    assert np.abs(f32(got.float().cpu()) - want).max() <= bar * max(1.0, np.abs(want).max() / 2)


@pytest.mark.parametrize("bh,sq,sk,d,dtype", [
    (3, 33, 8, 64, "fp16"), (2, 31, 64, 128, "bf16"), (9, 32, 65, 128, "fp16"), (2, 65, 129, 64, "fp16"), (17, 40, 191, 64, "bf16"),
    (2, 100, 333, 128, "fp16"), (2, 48, 448, 128, "fp16"), (2, 64, 511, 64, "fp16"), (2, 96, 640, 64, "bf16"),
])
def test_blocks_of_64_keys(bh, sq, sk, d, dtype, monkeypatch):
    monkeypatch.setenv("FMHA_FWD_COLS", "1")
    q, k, v = make_qkv(bh, sq, sk, d, seed=sk + d, dtype=dtype)
    g = torch.Generator().manual_seed(sk)
    m = (torch.rand(bh, sq, sk, generator=g) < 0.3).to(TDT[dtype]) * -1000
    m[:, 5] = float("-inf")                     # a row without a visible key
    m[:, 6, :-1] = float("-inf")                # one with the last key only
    dm = (torch.rand(bh, sq, sk, generator=g) < 0.5).to(TDT[dtype])
    bar, unit = BAR[dtype]
    qc, kc, vc, mc, dc = (t.cuda() for t in (q, k, v, m, dm))
    ref = oracle.attention(f32(q), f32(k), f32(v), mask=f32(m), want=("o", "lse"))
    o, lse, _, _ = capi.fwd(qc, kc, vc, mask=mc, want_lse=True)
    _check(o, ref["o"], bar)
    lse = lse.cpu().numpy()
    assert np.array_equal(np.isneginf(lse), np.isneginf(ref["lse"]))
    live = np.isfinite(ref["lse"])
    assert np.abs(lse[live] - ref["lse"][live]).max() <= 1e-3 + unit * np.abs(ref["lse"][live]).max()
    kw = dict(mask=mc, drop_kind=capi.DROP_TENSOR, drop_mask=dc, drop_scale=2.0)
    plain = capi.fwd(qc, kc, vc, **kw)[0]
    saved = capi.fwd(qc, kc, vc, save=True, **kw)
    assert torch.equal(saved[0], plain)
    s = torch.einsum("bqd,bkd->bqk", q.double(), k.double()) * d ** -0.5 + m.double()
    p = torch.softmax(s, -1).nan_to_num(0.0)
    _check(plain, (p * dm.double() * 2) .matmul(v.double()).numpy(), 2 * bar)
    _check(saved[2], p.numpy(), bar / 2)
    _check(saved[3], (p * dm.double() * 2).numpy(), bar)


@pytest.mark.parametrize("op,bh,s,d", [("infer", 16, 512, 64), ("infer", 17, 512, 64), ("train", 32, 500, 64), ("train", 33, 500, 64),
                                       ("train", 8, 64, 128), ("infer", 8, 65, 128), ("train", 8, 128, 64), ("train", 4, 449, 128)])
def test_few_workgroups_of_the_operators(op, bh, s, d, monkeypatch):
    """The operators take this kernel up to one workgroup per compute unit, with a dropout tensor two (256 of them on this device)."""
    monkeypatch.delenv("FMHA_FWD_COLS", raising=False)
    ops = load_ops()
    q, k, v = (t.cuda() for t in make_qkv(bh, s, s, d, seed=s))
    keep = (torch.rand(bh, s, s, device="cuda") < 0.9).half()
    args = (q, k, v, keep) if op == "infer" else (q, k, v, (1 - keep) * -1000, (torch.rand(bh, s, s, device="cuda") < 0.5).half())
    call = ops.fmha_nvfuser if op == "infer" else ops.fmha_train_nvfuser
    got = {}
    for env in (None, "0", "1"):
        if env:
            monkeypatch.setenv("FMHA_FWD_COLS", env)
        capi.lib().fmha_reload_overrides()
        got[env] = call(*args)
    monkeypatch.delenv("FMHA_FWD_COLS")
    capi.lib().fmha_reload_overrides()
    here = bh * ((s + 31) // 32) <= (256 if op == "infer" else 512) and (128 if d == 64 else 64) < s <= (640 if d == 64 else 448)
    assert torch.equal(got[None], got["1" if here else "0"])
    assert (got["0"].float() - got["1"].float()).abs().max() <= 4e-3
