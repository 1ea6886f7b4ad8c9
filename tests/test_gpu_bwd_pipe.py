"""The software-pipelined backward kernels at the edges of their tiles, segments and pipelines, against the CPU oracle:
one to a few 32-row tiles, ragged ends, more than one segment of staged queries (1024) and mask terms (4096), causal
heads whose keys outnumber the queries and the other way round."""
import pytest
import torch

import oracle
from nvfuserexamples_amd import capi
from conftest import f32, make_qkv, pad_mask, rel_to_max

pytestmark = pytest.mark.gpu

TDT = {"fp16": torch.float16, "bf16": torch.bfloat16}
TOL = {"fp16": 1e-2, "bf16": 3e-2}

CASES = [
    # bh, sq, sk, d, dtype, pad mask, causal, p
    (2, 1, 300, 64, "fp16", False, False, 0.1),
    (2, 300, 1, 64, "fp16", False, False, 0.0),
    (2, 257, 33, 64, "bf16", True, False, 0.1),
    (2, 31, 289, 64, "fp16", True, True, 0.1),
    (2, 290, 64, 64, "fp16", False, True, 0.0),
    (1, 33, 33, 128, "fp16", False, False, 0.1),
    (1, 96, 128, 128, "bf16", True, True, 0.0),
    (1, 130, 97, 128, "fp16", False, True, 0.1),
    (2, 161, 95, 96, "fp16", True, False, 0.1),       # columns that rows do not have
    (1, 1100, 96, 64, "fp16", False, False, 0.1),     # queries in two segments
    (1, 2081, 40, 128, "fp16", False, False, 0.1),    # ... in three
    (1, 1056, 1056, 128, "bf16", False, True, 0.1),   # ... under a causal mask
    (1, 40, 4200, 64, "fp16", True, False, 0.0),      # mask terms in two segments
]


@pytest.mark.parametrize("bh,sq,sk,d,dtype,pad,causal,p", CASES)
def test_pipelined_backward_at_its_edges(bh, sq, sk, d, dtype, pad, causal, p):
    q, k, v, do = make_qkv(bh, sq, sk, d, seed=sq + sk, std=0.7, dtype=dtype, with_dout=True)
    m = pad_mask(1, sk, max(1, sk // 2), sk, seed=5).to(TDT[dtype]) if pad else None
    kw = dict(causal=causal)
    okw = dict(causal=causal)
    if p > 0:
        kw.update(drop_kind=capi.DROP_PHILOX, p_drop=p, seed=99, offset=12)
        okw.update(philox=True, p_drop=p, seed=99, offset=12)
    qc, kc, vc, mc = q.cuda(), k.cuda(), v.cuda(), (None if m is None else m.cuda())
    o, lse, _, _ = capi.fwd(qc, kc, vc, mask=mc, want_lse=True, **kw)
    got = capi.bwd(do.cuda(), qc, kc, vc, o, lse, mask=mc, **kw)
    torch.cuda.synchronize()
    ref = oracle.attention(f32(q), f32(k), f32(v), mask=None if m is None else f32(m), dout=f32(do),
                           want=("dq", "dk", "dv"), **okw)
    for name, t in zip(("dq", "dk", "dv"), got):
        assert rel_to_max(f32(t.cpu()), ref[name], floor=1e-2) <= TOL[dtype], name


@pytest.mark.parametrize("bh,sq,sk,dtype,pad,p", [(3, 129, 300, "bf16", False, 0.0), (2, 384, 384, "fp16", False, 0.0), (2, 400, 333, "bf16", True, 0.1),
                                                  (1, 895, 900, "fp16", False, 0.1), (1, 896, 896, "fp16", True, 0.0)])
def test_causal_pairs_at_head_dim_128(bh, sq, sk, dtype, pad, p, monkeypatch):
    """Pairs of causal tiles, as launches of many heads have them: two query tiles and up, even and odd numbers of them, the
    second tile of a pair on lane constants that are set up anew.  (The kernels phase by phase take pairs under full mask tensors
    only: test_causal_tile_pairing_under_a_full_mask.)"""
    monkeypatch.setenv("FMHA_BWD_PAIR", "1")
    capi.lib().fmha_reload_overrides()
    try:
        test_pipelined_backward_at_its_edges(bh, sq, sk, 128, dtype, pad, True, p)
    finally:
        monkeypatch.delenv("FMHA_BWD_PAIR")
        capi.lib().fmha_reload_overrides()


@pytest.mark.parametrize("sq,sk,d,dtype,live,p", [
    (4097, 4097, 64, "fp16", 4097, 0.1),    # the smallest: one key and one query in the second segment
    (4480, 4480, 64, "fp16", 3000, 0.0),    # every live key in the first segment, the second all hard-masked
    (4480, 4480, 64, "bf16", 4300, 0.1),
    (4300, 4128, 96, "fp16", 4128, 0.0),    # run-time rows with columns that do not exist
    (4224, 4480, 128, "fp16", 2500, 0.1),
    (4480, 4480, 128, "bf16", 4400, 0.0),
    (8320, 8320, 64, "fp16", 8200, 0.0),    # three segments (both forms of the launch against each other only)
])
def test_causal_pairs_read_the_mask_terms_of_their_own_segment(sq, sk, d, dtype, live, p, monkeypatch):
    """Pairs of causal query tiles under a per-key mask of more than 4096 keys: the first tile of a pair leaves the mask
    terms of its last segment behind, the second one starts at key 0 again.  Distinct terms for every key and a hard-masked
    tail; gradients against the oracle, and the same bits as without pairs (a tile's arithmetic does not depend on them)."""
    q, k, v, do = make_qkv(1, sq, sk, d, seed=sq + sk, std=0.7, dtype=dtype, with_dout=True)
    m = -2.0 * torch.rand(1, 1, 1, sk, generator=torch.Generator().manual_seed(3))
    m[..., live:] = -10000.0
    m = m.to(TDT[dtype])
    kw, okw = dict(causal=True), dict(causal=True)
    if p > 0:
        kw.update(drop_kind=capi.DROP_PHILOX, p_drop=p, seed=99, offset=12)
        okw.update(philox=True, p_drop=p, seed=99, offset=12)
    dev = [t.cuda() for t in (q, k, v, do, m)]
    o, lse, _, _ = capi.fwd(*dev[:3], mask=dev[4], want_lse=True, **kw)
    got = {}
    try:
        for pair in ("0", "1"):
            monkeypatch.setenv("FMHA_BWD_PAIR", pair)
            capi.lib().fmha_reload_overrides()
            got[pair] = capi.bwd(dev[3], *dev[:3], o, lse, mask=dev[4], **kw)
            torch.cuda.synchronize()
    finally:
        monkeypatch.delenv("FMHA_BWD_PAIR")
        capi.lib().fmha_reload_overrides()
    for name, a, b in zip(("dq", "dk", "dv"), got["0"], got["1"]):
        assert torch.equal(a, b), name
    if sk > 8192:
        return
    ref = oracle.attention(f32(q), f32(k), f32(v), mask=f32(m), dout=f32(do), want=("dq", "dk", "dv"), **okw)
    for name, t in zip(("dq", "dk", "dv"), got["1"]):
        assert rel_to_max(f32(t.cpu()), ref[name], floor=1e-2) <= TOL[dtype], name
