"""Head dims up to 32 and from 72 to 96: kernels of their own widths (32 and 96) on LDS tiles of whole 64-column panels.

Lengths around the 32-row blocks, the 64- and 128-row tiles and the lines between kernels; whole rows and rows that end before the
width; a full mask tensor, which the next whole panel's kernels take.  Oracle and bars of ``test_gpu_head_dims.py``.
"""
import numpy as np
import pytest
import torch

import oracle
from nvfuserexamples_amd import capi
from conftest import make_qkv, pad_mask, f32, rel_to_max

pytestmark = pytest.mark.gpu

TDT = {"fp16": torch.float16, "bf16": torch.bfloat16}
O_TOL = {"fp16": 2e-3, "bf16": 2e-2}
G_TOL = {"fp16": 1e-2, "bf16": 3e-2}

CASES = [
    # bh, sq, sk, d, dtype, causal, p_drop, mask
    (2, 31, 33, 32, "fp16", False, 0.0, None),
    (2, 33, 31, 96, "bf16", False, 0.0, "pad"),
    (2, 127, 129, 96, "fp16", False, 0.1, None),
    (2, 129, 127, 32, "bf16", True, 0.1, None),
    (4, 257, 191, 72, "fp16", False, 0.0, "pad"),
    (4, 193, 257, 24, "fp16", False, 0.1, "pad"),
    (3, 385, 385, 80, "bf16", True, 0.0, None),
    (2, 900, 900, 96, "fp16", True, 0.1, None),
    (2, 1030, 1030, 32, "fp16", True, 0.0, None),   # extra-step rows in two segments
    (160, 260, 260, 32, "fp16", True, 0.0, None),   # more workgroups than are resident together
    (160, 260, 260, 96, "bf16", False, 0.1, "pad"),
    (160, 260, 260, 88, "fp16", True, 0.0, None),
    (2, 130, 150, 96, "fp16", False, 0.0, "full"),
    (2, 130, 150, 32, "bf16", False, 0.1, "full"),
]


@pytest.mark.parametrize("split", [False, True], ids=["", "split"])
@pytest.mark.parametrize("bh,sq,sk,d,dtype,causal,p,mask", CASES)
def test_widths_between_whole_panels(bh, sq, sk, d, dtype, causal, p, mask, split):
    q, k, v, do = make_qkv(bh, sq, sk, d, seed=3 * d + sq, dtype=dtype, with_dout=True)
    m = None
    if mask == "pad":
        m = pad_mask(2, sk, sk // 2, sk).to(TDT[dtype]) if bh % 2 == 0 else pad_mask(1, sk, sk // 2, sk).to(TDT[dtype])
    elif mask == "full":
        m = torch.randn(bh, sq, sk, generator=torch.Generator().manual_seed(d)).to(TDT[dtype])
    kw, okw = dict(causal=causal, scale=d ** -0.5), dict(causal=causal)
    if m is not None:
        kw["mask"] = m.cuda()
    if p:
        kw.update(drop_kind=capi.DROP_PHILOX, p_drop=p, seed=9, offset=4)
        okw.update(philox=True, p_drop=p, seed=9, offset=4)
    fkw = dict(kw, flags=4) if split else kw  # FMHA_FLAG_SPLIT_KEYS: the forward whose waves share 32 queries
    qc, kc, vc, doc = q.cuda(), k.cuda(), v.cuda(), do.cuda()
    o, lse, _, _ = capi.fwd(qc, kc, vc, want_lse=True, **fkw)
    dq, dk, dv = capi.bwd(doc, qc, kc, vc, o, lse, **kw)
    torch.cuda.synchronize()
    ref = oracle.attention(f32(q), f32(k), f32(v), mask=None if m is None else f32(m), dout=f32(do),
                           want=("o", "lse", "dq", "dk", "dv"), **okw)
    assert np.abs(f32(o.cpu()) - ref["o"]).max() <= O_TOL[dtype]
    assert np.abs(lse.cpu().numpy() - ref["lse"]).max() <= (2e-3 if dtype == "fp16" else 1e-2)
    for name, g in (("dq", dq), ("dk", dk), ("dv", dv)):
        assert rel_to_max(f32(g.cpu()), ref[name], floor=1e-3) <= G_TOL[dtype], name


@pytest.mark.parametrize("d", [24, 80])
def test_infinite_keys_of_no_weight_do_not_reach_the_columns_a_row_lacks(d):
    """A key of -infinity in its first column has weight 0 for queries that are positive there, in the columns behind d too."""
    bh, s = 2, 160
    q, k, v = make_qkv(bh, s, s, d, seed=d)
    q[..., 0] = q[..., 0].abs() + 0.5
    k[:, 37, 0] = float("-inf")
    got = capi.fwd(q.cuda(), k.cuda(), v.cuda(), scale=d ** -0.5)[0]
    keep = [i for i in range(s) if i != 37]
    ref = oracle.attention(f32(q), f32(k[:, keep]), f32(v[:, keep]), want=("o",))
    assert np.abs(f32(got.cpu()) - ref["o"]).max() <= O_TOL["fp16"]
