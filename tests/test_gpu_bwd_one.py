"""The one-pass backward (head dim 64, 129 to 256 queries or keys, more heads than the device holds at once) at the edges of its
tiles, against the launches of few heads, which run on the kernel for short heads (compared with the oracle in test_gpu_bwd.py).

Both kernels keep scores and sums in fp32 and round P, dS and the gradients to the element type (u = 2^-11 in fp16, 2^-8 in
bf16).  Their P and dS before rounding differ by a few ulp of fp32, so a rounding may fall the other way, which moves a term by
up to 2 u of itself.  A gradient is a sum of terms of either sign: such moves add up like the terms do, to 2 u of a gradient's
own size, and the result's rounding may turn as well: 4 u max|gradient|.  With dropout the heads behind the first 250 cannot be
launched by themselves (decisions go by a head's number); all heads are compared with the two general kernels there, which
also round Q * scale: scores off by u of themselves, |score| < 6 for nearly all of P, so twice the bound.
"""
import pytest
import torch

from nvfuserexamples_amd import capi
from conftest import make_qkv, tail_mask

pytestmark = pytest.mark.gpu

TDT = {"fp16": torch.float16, "bf16": torch.bfloat16}
U = {"fp16": 2.0 ** -11, "bf16": 2.0 ** -8}
HPR = 10  # heads per mask row / key count

CASES = [
    # bh, sq, sk, dtype, mask, causal, p, packed
    (520, 129, 129, "fp16", None, False, 0.0, False),    # a fifth tile of one row, a wave of one key; two heads a workgroup and more
    (260, 1, 129, "fp16", None, False, 0.1, False),      # one query tile: three turns of padding, heads right behind one another
    (300, 40, 256, "bf16", None, True, 0.0, False),      # two query tiles; keys behind every query
    (300, 256, 33, "fp16", None, False, 0.1, False),     # a wave of one key, six of none
    (1030, 96, 160, "fp16", "len", False, 0.0, False),   # three query tiles; key counts, among them 0; five heads a workgroup
    (270, 256, 256, "bf16", "tail", False, 0.1, True),   # packed rows
    (270, 197, 197, "fp16", "inf", True, 0.1, False),    # -inf in the mask
    (270, 224, 225, "fp16", "lowest", False, 0.0, True),  # the type's lowest value in the mask
    (270, 200, 140, "bf16", "lowest", True, 0.1, True),
    (270, 160, 250, "fp16", "dead", False, 0.1, False),  # rows that see no key
]


@pytest.mark.parametrize("bh,sq,sk,dtype,mask,causal,p,packed", CASES)
def test_one_pass_matches_the_kernel_for_short_heads(bh, sq, sk, dtype, mask, causal, p, packed, monkeypatch):
    q, k, v, do = (t.cuda() for t in make_qkv(bh, sq, sk, 64, seed=sq + sk, std=1.0, dtype=dtype, with_dout=True))
    rows = bh // HPR
    m = lens = None
    g = torch.Generator().manual_seed(7)
    if mask == "len":
        lens = torch.randint(0, sk + 1, (rows,), generator=g, dtype=torch.int32)
        lens[1] = 0
        lens[-1] = sk
        lens = lens.cuda()
    elif mask == "tail":
        m = tail_mask(mask, rows, sk, seed=11)
    elif mask:
        m = torch.randn(rows, 1, sk, generator=g)
        m[:, :, 3::5] = float("-inf") if mask != "lowest" else torch.finfo(TDT[dtype]).min
        if mask == "dead":
            m[2] = float("-inf")
    m = None if m is None else m.to(TDT[dtype]).cuda()
    kw = dict(causal=causal)
    if p > 0:
        kw.update(drop_kind=capi.DROP_PHILOX, p_drop=p, seed=99, offset=12)

    def args(h0, h1):
        r = slice(h0 // HPR, h1 // HPR)
        return dict(kw, mask=None if m is None else m[r], kv_len=None if lens is None else lens[r])

    def rows_apart(t):  # [bh, s, 64] -> the same values, the rows of HPR heads beside each other
        return t.view(bh // HPR, HPR, t.shape[1], 64).transpose(1, 2).contiguous().transpose(1, 2)

    o, lse, _, _ = capi.fwd(q, k, v, want_lse=True, **args(0, bh))
    ins = [rows_apart(t) for t in (do, q, k, v, o)] if packed else [do, q, k, v, o]
    fill = [torch.full_like(t, 7.0) for t in ins[1:4]]  # (every element has to be written)
    capi.bwd(*ins, lse, grads=tuple(fill), **args(0, bh))
    got = [t.reshape(bh, t.shape[-2], 64) for t in fill]

    def close(h0, h1, ref, terms):
        for name, a, b in zip(("dq", "dk", "dv"), got, ref):
            a, b = a[h0:h1].float(), b.float()
            assert torch.isfinite(a).all() and torch.isfinite(b).all(), name
            assert (a - b).abs().max().item() <= terms * U[dtype] * b.abs().max().item() + 1e-6, name

    for h0 in (0,) if p > 0 else (0, bh - 250):
        few = [t[h0:h0 + 250].contiguous() for t in (do, q, k, v, o, lse)]
        close(h0, h0 + 250, capi.bwd(*few, **args(h0, h0 + 250)), 4)
    if p > 0:
        monkeypatch.setenv("FMHA_BWD_SHORT", "0")
        capi.lib().fmha_reload_overrides()
        try:
            close(0, bh, capi.bwd(do, q, k, v, o, lse, **args(0, bh)), 8)
        finally:
            monkeypatch.undo()
            capi.lib().fmha_reload_overrides()
    assert not any((t == 7.0).all(-1).any() for t in got)
