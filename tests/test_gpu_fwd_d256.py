"""The pipelined forward at head dim 256 (and the head dims that run on it): tile edges, items that follow one another in a
workgroup, masks, key counts, dropout, run-time rows.  Bars as in test_gpu_fwd.py: 2e-3 for fp16 and 2e-2 for bf16 on O (P and O
are rounded to the element type, Q * scale once before the first product); LSE within 2^-11 / 2^-8 of the scores' own size
(|score| < 8 here) and of the row sum, which is that of the rounded P."""
import numpy as np
import pytest
import torch

import oracle
from nvfuserexamples_amd import capi
from conftest import make_qkv, tail_mask, f32

pytestmark = pytest.mark.gpu

TOL = {"fp16": 2e-3, "bf16": 2e-2}
U = {"fp16": 2.0 ** -11, "bf16": 2.0 ** -8}
TDT = {"fp16": torch.float16, "bf16": torch.bfloat16}
HPR = 4  # heads per mask row / key count

CASES = [
    # bh, sq, sk, d, dtype, mask, causal, p, packed
    (4, 128, 64, 256, "fp16", None, False, 0.0, False),      # one tile: the plain loop
    (4, 1, 65, 256, "fp16", None, False, 0.0, False),        # a second tile of one key
    (4, 129, 128, 256, "bf16", None, False, 0.1, False),
    (4, 300, 193, 256, "fp16", "inf", True, 0.0, True),
    (4, 130, 320, 256, "fp16", "tail", False, 0.1, False),
    (8, 200, 200, 256, "bf16", "len", True, 0.0, True),      # key counts, among them 0
    (264, 100, 130, 256, "fp16", "len", False, 0.0, False),  # two items a workgroup
    (132, 300, 300, 256, "bf16", None, True, 0.1, False),    # three query tiles a head, heads in two rounds
    (264, 70, 257, 256, "fp16", "some_rows_all_masked", False, 0.0, False),
    (4, 160, 129, 136, "fp16", None, False, 0.0, False),     # head dims that are filled up
    (132, 200, 200, 200, "bf16", "tail", True, 0.0, True),
]


@pytest.mark.parametrize("bh,sq,sk,d,dtype,mask,causal,p,packed", CASES)
def test_forward_at_head_dim_256(bh, sq, sk, d, dtype, mask, causal, p, packed):
    q, k, v = make_qkv(bh, sq, sk, d, seed=sq + sk, std=0.5, dtype=dtype)[:3]
    v = (v * 2).to(TDT[dtype])
    rows = bh // HPR
    m = lens = None
    if mask == "len":
        lens = torch.randint(0, sk + 1, (rows,), generator=torch.Generator().manual_seed(7), dtype=torch.int32)
        lens[0], lens[-1] = 0, sk
    elif mask:
        m = tail_mask(mask, rows, sk, seed=11).to(TDT[dtype])
    kw = dict(causal=causal)
    if p > 0:
        kw.update(drop_kind=capi.DROP_PHILOX, p_drop=p, seed=99, offset=12)

    def dev(t):  # (packed: the rows of HPR heads beside each other)
        t = t.cuda()
        return t.view(rows, HPR, t.shape[1], d).transpose(1, 2).contiguous().transpose(1, 2) if packed else t

    o, lse, _, _ = capi.fwd(dev(q), dev(k), dev(v), mask=None if m is None else m.cuda(), want_lse=True,
                            kv_len=None if lens is None else lens.cuda(), **kw)
    torch.cuda.synchronize()
    o, lse = f32(o.reshape(bh, sq, d).cpu()), lse.cpu().numpy().reshape(bh, sq)
    assert np.isfinite(o).all()
    for h in sorted({0, 1, bh // 2, bh - HPR, bh - 1}):
        mo = None if m is None else f32(m[h // HPR]).reshape(1, 1, sk)
        if lens is not None:
            mo = np.zeros((1, 1, sk), np.float32)
            mo[..., int(lens[h // HPR]):] = -np.inf
        okw = dict(philox=True, p_drop=p, seed=99, offset=12, bh_offset=h) if p > 0 else {}
        ref = oracle.attention(f32(q[h:h + 1]), f32(k[h:h + 1]), f32(v[h:h + 1]), mask=mo, causal=causal,
                               want=("o", "lse"), **okw)
        assert np.abs(o[h] - ref["o"][0]).max() <= TOL[dtype], h
        a, b = lse[h], np.asarray(ref["lse"]).reshape(sq)
        live = np.isfinite(b)
        assert (np.isneginf(a) == ~live).all()
        big = np.maximum(8, np.abs(b[live]))  # (a row under a finite mask: its scores are that large)
        assert (np.abs(a[live] - b[live]) <= 2 * U[dtype] * big).all(), h
