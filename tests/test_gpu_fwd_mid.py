"""The forward for 129 to 256 keys (head dim 64, a head's K and V in LDS) at the edges of its blocks and of its dispatch: workgroups
of four waves while each has a compute unit to itself, of eight beyond.

Bound: scores, exponents and sums are fp32; P is rounded once to the element type (relative error u = 2^-11, bf16 2^-8) and so is
O.  With rows of P that sum to one, times the dropout factor f, |O - oracle| <= 2 u f max|V|, and 1e-5 for the fp32 steps.  The
row sum is that of the rounded P: the log-sum-exp is off by up to u, and 1e-5 of its size for the fp32 steps."""
import numpy as np
import pytest
import torch

import oracle
from nvfuserexamples_amd import capi
from conftest import make_qkv, f32

pytestmark = pytest.mark.gpu

TDT = {"fp16": torch.float16, "bf16": torch.bfloat16}
U = {"fp16": 2.0 ** -11, "bf16": 2.0 ** -8}
HPR = 4  # heads per mask row / key count

CASES = [
    # bh, sq, sk, dtype, mask, causal, p, packed
    (8, 129, 129, "fp16", None, False, 0.0, False),      # four waves: a block of one key, a wave of one query
    (4, 300, 192, "bf16", "len", False, 0.0, False),     # three workgroups a head; key counts, among them 0
    (8, 256, 256, "fp16", "inf", True, 0.1, False),
    (8, 160, 225, "fp16", "lowest", False, 0.1, False),  # the type's lowest value; more than seven blocks
    (8, 200, 200, "bf16", "dead", True, 0.0, True),      # rows that see no key
    (4, 600, 140, "fp16", "rising", False, 0.0, False),  # the reference is raised in every block
    (8, 129, 256, "fp16", None, True, 0.1, False),       # keys behind every query
    (264, 129, 129, "fp16", None, False, 0.1, False),    # eight waves
    (264, 257, 161, "bf16", "len", True, 0.0, True),     # a second workgroup with one query
    (264, 256, 224, "fp16", "rising", True, 0.1, False),
    (264, 197, 197, "bf16", None, False, 0.0, True),
    (1032, 256, 256, "fp16", "inf", False, 0.0, False),  # eight blocks without dropout: from four workgroups a compute unit on
    (264, 250, 255, "bf16", "lowest", False, 0.1, True),
]


@pytest.mark.parametrize("bh,sq,sk,dtype,mask,causal,p,packed", CASES)
def test_forward_of_129_to_256_keys(bh, sq, sk, dtype, mask, causal, p, packed):
    q, k, v = make_qkv(bh, sq, sk, 64, seed=sq + sk, dtype=dtype)[:3]
    rows, g = bh // HPR, torch.Generator().manual_seed(7)
    m = lens = None
    if mask == "len":
        lens = torch.randint(0, sk + 1, (rows,), generator=g, dtype=torch.int32)
        lens[0], lens[-1] = 0, sk
    elif mask == "rising":
        m = torch.arange(sk).float().mul(0.4).expand(rows, 1, sk).clone()
    elif mask:
        m = torch.randn(rows, 1, sk, generator=g)
        m[:, :, 3::5] = float("-inf") if mask != "lowest" else torch.finfo(TDT[dtype]).min
        m[0, :, sk // 2:] = float("-inf")
        if mask == "dead":
            m[-1] = float("-inf")
    m = None if m is None else m.to(TDT[dtype])
    kw = dict(causal=causal)
    if p > 0:
        kw.update(drop_kind=capi.DROP_PHILOX, p_drop=p, seed=99, offset=12)

    def dev(t):  # (packed: the rows of HPR heads beside each other)
        t = t.cuda()
        return t.view(rows, HPR, t.shape[1], 64).transpose(1, 2).contiguous().transpose(1, 2) if packed else t

    o, lse, _, _ = capi.fwd(dev(q), dev(k), dev(v), mask=None if m is None else m.cuda(), want_lse=True,
                            kv_len=None if lens is None else lens.cuda(), **kw)
    torch.cuda.synchronize()
    o, lse = f32(o.reshape(bh, sq, 64).cpu()), lse.cpu().numpy().reshape(bh, sq)
    assert np.isfinite(o).all()
    for h in sorted({0, 1, bh // 2, bh - HPR, bh - 1}):
        mo = None if m is None else f32(m[h // HPR]).reshape(1, 1, sk)
        if lens is not None:
            mo = np.zeros((1, 1, sk), np.float32)
            mo[..., int(lens[h // HPR]):] = -np.inf
        okw = dict(philox=True, p_drop=p, seed=99, offset=12, bh_offset=h) if p > 0 else {}
        ref = oracle.attention(f32(q[h:h + 1]), f32(k[h:h + 1]), f32(v[h:h + 1]), mask=mo, causal=causal,
                               want=("o", "lse"), **okw)
        f = 1 / (1 - round(256 * p) / 256)
        assert np.abs(o[h] - ref["o"][0]).max() <= 2 * U[dtype] * f * np.abs(f32(v[h])).max() + 1e-5, h
        a, b = lse[h], np.asarray(ref["lse"]).reshape(sq)
        live = np.isfinite(b)
        assert (np.isneginf(a) == ~live).all()
        assert (np.abs(a[live] - b[live]) <= U[dtype] + 1e-5 * np.maximum(1, np.abs(b[live]))).all(), h
