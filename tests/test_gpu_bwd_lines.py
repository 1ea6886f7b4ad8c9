"""The backward on both sides of the lines where its kernels change, with ragged last tiles and numbers of heads that do not divide
over the compute dies: causal dQ at head dim 128 (pipelined from 128 queries on), dK / dV at head dim 128 under masks and key counts
without dropout (from 192, of shorter rows from 385), heads left over behind groups of eight, dQ at head dims up to 96 whose products
start from LSE and delta (only a mask has an extra step: the last tile's missing keys are a test per score), rows narrower than the kernel's, against the oracle."""
import numpy as np
import pytest
import torch

import oracle
from conftest import f32, make_qkv, pad_mask
from nvfuserexamples_amd import capi

pytestmark = pytest.mark.gpu

TDT = {"fp16": torch.float16, "bf16": torch.bfloat16}
UNIT = {"fp16": 2.0 ** -11, "bf16": 2.0 ** -8}  # one rounding of a value to the element type

CASES = [
    # bh, sq, sk, d, dtype, mask, causal, p
    (3, 127, 127, 128, "fp16", None, True, 0.0),
    (9, 128, 128, 128, "bf16", None, True, 0.1),
    (3, 129, 161, 128, "fp16", "pad", True, 0.1),
    (2, 225, 97, 112, "bf16", "len", True, 0.0),
    (2, 415, 415, 128, "fp16", None, True, 0.1),
    (3, 191, 65, 128, "bf16", "pad", False, 0.0),
    (9, 192, 193, 128, "fp16", "len", False, 0.0),
    (11, 193, 31, 128, "bf16", "pad", False, 0.0),
    (3, 384, 129, 104, "fp16", "pad", False, 0.0),
    (3, 385, 129, 104, "fp16", "len", False, 0.0),
    (13, 70, 333, 64, "fp16", "pad", False, 0.1),  # five heads left over behind the eight of a group
    (12, 385, 300, 64, "fp16", "len", False, 0.0),  # the four left over are ranges of each die
    (20, 260, 257, 128, "bf16", "pad", False, 0.1),
    (7, 300, 400, 96, "bf16", "pad", False, 0.0),   # fewer than eight heads
    (3, 257, 289, 64, "fp16", None, False, 0.0),
    (9, 257, 290, 64, "bf16", "len", False, 0.1),
    (3, 300, 287, 64, "bf16", None, True, 0.1),
    (2, 290, 321, 96, "fp16", None, False, 0.0),
    (3, 257, 299, 80, "bf16", "len", True, 0.0),
    (5, 300, 299, 32, "fp16", "len", True, 0.1),
    (3, 129, 161, 32, "bf16", None, False, 0.0),
    (3, 70, 100, 48, "fp16", "pad", False, 0.1),   # narrow rows one behind the other: register operands loaded as wanted
    (2, 290, 257, 40, "bf16", None, False, 0.0),
    (2, 201, 230, 56, "fp16", "len", True, 0.1),   # ... and turned
]


@pytest.mark.parametrize("bh,sq,sk,d,dtype,mask,causal,p", CASES)
def test_backward_on_both_sides_of_its_lines(bh, sq, sk, d, dtype, mask, causal, p):
    q, k, v, do = make_qkv(bh, sq, sk, d, seed=sq + sk + d, std=0.7, dtype=dtype, with_dout=True)
    kw, okw, m, om = dict(causal=causal), dict(causal=causal), None, None
    if mask == "pad":
        m = pad_mask(1, sk, max(1, sk // 2), sk, seed=5).to(TDT[dtype])
        om = f32(m)
    elif mask == "len":
        n = sk - sk // 3
        kw["kv_len"] = torch.tensor([n], dtype=torch.int32, device="cuda")
        om = f32(torch.where(torch.arange(sk) < n, 0.0, float("-inf")).view(1, 1, sk))
    if p > 0:
        kw.update(drop_kind=capi.DROP_PHILOX, p_drop=p, seed=99, offset=12)
        okw.update(philox=True, p_drop=p, seed=99, offset=12)
    qc, kc, vc, mc = q.cuda(), k.cuda(), v.cuda(), (None if m is None else m.cuda())
    o, lse, _, _ = capi.fwd(qc, kc, vc, mask=mc, want_lse=True, **kw)
    got = capi.bwd(do.cuda(), qc, kc, vc, o, lse, mask=mc, **kw)
    torch.cuda.synchronize()
    ref = oracle.attention(f32(q), f32(k), f32(v), mask=om, dout=f32(do), want=("dq", "dk", "dv"), **okw)
    # P, dS, O (in delta) and the result are rounded once each, by one unit of their size at most, and dP - delta may lose part of its
    # size to the subtraction: twice the four units bound the norm of the error.
    for name, t in zip(("dq", "dk", "dv"), got):
        assert np.linalg.norm(f32(t.cpu()) - ref[name]) <= 8 * UNIT[dtype] * np.linalg.norm(ref[name]), name


MASKED = [
    # b, h, sq, sk, dtype, mask, packed: dK / dV at head dim 128 without dropout and causal mask, pipelined
    (3, 2, 1056, 130, "fp16", "pad", False),   # rows (-LSE, -delta) in two segments
    (3, 1, 1100, 1100, "bf16", "len", True),
    (2, 4, 200, 200, "fp16", "pad", True),
    (4, 3, 192, 257, "bf16", "len", False),
]


@pytest.mark.parametrize("b,h,sq,sk,dtype,mask,packed", MASKED)
def test_masked_dk_dv_at_head_dim_128(b, h, sq, sk, dtype, mask, packed):
    """More than one segment of queries, packed rows, and lengths that differ between the sequences: none, one key, half, all."""
    d = 128
    q, k, v, do = make_qkv(b * h, sq, sk, d, seed=sq + sk, std=0.7, dtype=dtype, with_dout=True)
    lens = [0 if mask == "len" else 2, sk, sk // 2, 1][:b]
    live = torch.arange(sk)[None] < torch.tensor(lens)[:, None]
    kw = dict(kv_len=torch.tensor(lens, dtype=torch.int32).cuda()) if mask == "len" else dict(mask=torch.where(live, 0.0, -10000.0).to(TDT[dtype]).view(b, 1, 1, sk).cuda())
    if packed:
        qkv = torch.stack([t.view(b, h, sq, d).transpose(1, 2) for t in (q, k, v)], 2).cuda()  # [B, S, 3, H, D]
        dev = [qkv[:, :, i].transpose(1, 2) for i in range(3)] + [do.view(b, h, sq, d).transpose(1, 2).contiguous().cuda().transpose(1, 2)]
    else:
        dev = [t.cuda() for t in (q, k, v, do)]
    o, lse, _, _ = capi.fwd(*dev[:3], want_lse=True, **kw)
    got = [f32(t.reshape(b * h, -1, d).cpu()) for t in capi.bwd(dev[3], *dev[:3], o, lse, **kw)]
    torch.cuda.synchronize()
    shown = live | (torch.tensor(lens) == 0)[:, None]  # (a sequence without keys: no gradient at all, below)
    om = torch.where(shown, 0.0, float("-inf")).repeat_interleave(h, 0).unsqueeze(1).expand(b * h, sq, sk).contiguous()
    ref = oracle.attention(f32(q), f32(k), f32(v), mask=f32(om), dout=f32(do), want=("dq", "dk", "dv"))
    for name, t in zip(("dq", "dk", "dv"), got):
        for i, n in enumerate(lens):
            a, r = t[i * h:(i + 1) * h], ref[name][i * h:(i + 1) * h]
            if n == 0:
                assert not a.any(), (name, i)
                continue
            if name != "dq":
                assert not a[:, n:].any(), (name, i)
            # the bound of the test above; with one key dS is what rounding leaves of dP = dO V, 0.7^2 sqrt(d), times Q or K, 0.7 sqrt(d)
            # a row, times the scale, over rows that add up at random
            floor = 0.7 ** 3 * d * d ** -0.5 * np.sqrt(h * sq) if n == 1 and name != "dv" else 0.0
            assert np.linalg.norm(a - r) <= 8 * UNIT[dtype] * max(np.linalg.norm(r), floor), (name, i)
