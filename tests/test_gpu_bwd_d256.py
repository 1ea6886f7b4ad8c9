"""dQ at head dim 256 on the pipelined kernel (from 128 queries on), beside the wave-pair dK / dV kernel: tile edges, masks, key
counts, causal pairs, dropout, run-time rows.  Bar as in test_gpu_bwd.py: 1e-2 (bf16 3e-2) of the largest gradient."""
import numpy as np
import pytest
import torch

import oracle
from nvfuserexamples_amd import capi
from conftest import make_qkv, tail_mask, f32, rel_to_max

pytestmark = pytest.mark.gpu

TOL = {"fp16": 1e-2, "bf16": 3e-2}
TDT = {"fp16": torch.float16, "bf16": torch.bfloat16}

CASES = [
    # bh, sq, sk, d, dtype, mask, causal, p, pairs of causal tiles
    (4, 127, 64, 256, "fp16", None, False, 0.0, None),       # phase by phase
    (4, 128, 33, 256, "fp16", None, False, 0.1, None),       # a second tile of one key
    (4, 129, 31, 256, "bf16", None, False, 0.0, None),       # one tile, a workgroup of one query
    (4, 300, 200, 256, "fp16", "tail", True, 0.1, "0"),
    (4, 420, 420, 256, "bf16", None, True, 0.0, "1"),        # pairs, an even number of tiles
    (2, 520, 520, 256, "fp16", None, True, 0.1, "1"),        # ... an odd one
    (4, 160, 270, 256, "fp16", "len", False, 0.0, None),     # key counts, among them 0
    (2, 130, 4200, 256, "fp16", "tail", False, 0.0, None),   # mask terms in two segments
    (4, 140, 96, 136, "bf16", None, False, 0.1, None),       # head dims that are filled up
    (4, 260, 260, 200, "fp16", "tail", True, 0.0, None),
]


@pytest.mark.parametrize("bh,sq,sk,d,dtype,mask,causal,p,pair", CASES)
def test_backward_at_head_dim_256(bh, sq, sk, d, dtype, mask, causal, p, pair, monkeypatch):
    q, k, v, do = make_qkv(bh, sq, sk, d, seed=sq + sk, std=0.35, dtype=dtype, with_dout=True)
    m = lens = None
    if mask == "len":
        lens = torch.tensor([0, sk // 2 + 1], dtype=torch.int32)
    elif mask:
        m = tail_mask(mask, 2, sk, seed=11).to(TDT[dtype])
    kw, okw = dict(causal=causal), dict(causal=causal)
    if p > 0:
        kw.update(drop_kind=capi.DROP_PHILOX, p_drop=p, seed=99, offset=12)
        okw.update(philox=True, p_drop=p, seed=99, offset=12)
    mo = None if m is None else f32(m)
    if lens is not None:
        mo = np.zeros((2, 1, 1, sk), np.float32)
        for i, n in enumerate(lens.tolist()):
            mo[i, 0, 0, n:] = -np.inf
        kw["kv_len"] = lens.cuda()
    qc, kc, vc, mc = q.cuda(), k.cuda(), v.cuda(), (None if m is None else m.cuda())
    try:
        if pair is not None:
            monkeypatch.setenv("FMHA_BWD_PAIR", pair)
            capi.lib().fmha_reload_overrides()
        o, lse, _, _ = capi.fwd(qc, kc, vc, mask=mc, want_lse=True, **kw)
        got = capi.bwd(do.cuda(), qc, kc, vc, o, lse, mask=mc, **kw)
        torch.cuda.synchronize()
    finally:
        if pair is not None:
            monkeypatch.delenv("FMHA_BWD_PAIR")
            capi.lib().fmha_reload_overrides()
    ref = oracle.attention(f32(q), f32(k), f32(v), mask=mo, dout=f32(do), want=("dq", "dk", "dv"), **okw)
    for name, t in zip(("dq", "dk", "dv"), got):
        g = f32(t.cpu())
        assert np.isfinite(g).all(), name
        assert rel_to_max(g, ref[name], floor=1e-3) <= TOL[dtype], name
