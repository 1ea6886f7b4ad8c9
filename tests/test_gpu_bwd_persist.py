"""The persistent dK / dV kernel (head dim 128, no mask, from one and a half rounds of workgroups on): what a workgroup hands from
item to item.  A head's gradients do not depend on the heads beside it, so a launch of many heads has to give the bits of
launches of few heads, which run on the plain pipelined kernel (compared with the oracle in test_gpu_bwd_pipe.py).  The cases
with a mask or key counts are those whose launches stay on the plain kernels.

Few causal heads of fewer than 192 queries run phase by phase, with other roundings of the scaled operands: scores
are off by u of themselves (u = 2^-11, bf16 2^-8; |score| < 6 for nearly all of P), and roundings of P, dS and the result may
fall the other way: errors of either sign that add up like the gradient's own terms do, 8 u max|gradient|."""
import pytest
import torch

from nvfuserexamples_amd import capi
from conftest import make_qkv, tail_mask

pytestmark = pytest.mark.gpu

TDT = {"fp16": torch.float16, "bf16": torch.bfloat16}
U = {"fp16": 2.0 ** -11, "bf16": 2.0 ** -8}
HPR = 10  # heads per mask row / key count

CASES = [
    # bh, sq, sk, d, dtype, mask, causal, p, pairs of causal tiles
    (600, 128, 128, 128, "fp16", None, False, 0.0, None),        # the smallest: four turns an item
    (600, 129, 70, 128, "bf16", None, False, 0.1, None),         # a key tile with dead waves, queries past the end
    (260, 130, 300, 128, "fp16", None, False, 0.1, None),        # three key tiles, an uneven last round
    (130, 200, 500, 96, "fp16", None, False, 0.0, None),         # columns that rows do not have
    (260, 130, 300, 128, "fp16", "tail", False, 0.1, None),
    (100, 160, 700, 128, "fp16", "len", False, 0.0, None),       # key counts, among them 0
    (200, 130, 260, 128, "fp16", None, True, 0.1, "0"),          # items of one query tile; key tiles behind every query
    (200, 288, 420, 128, "fp16", None, True, 0.1, "0"),          # ... to the bit
    (400, 420, 420, 128, "bf16", None, True, 0.0, "1"),          # pairs, an even and (next) an odd number of tiles
    (400, 300, 300, 128, "fp16", None, True, 0.1, "1"),
    (200, 420, 420, 128, "bf16", None, True, 0.1, "0"),          # rounds in turned order
    (70, 700, 760, 80, "fp16", None, True, 0.0, "0"),
    (130, 1088, 400, 128, "fp16", None, False, 0.1, None),       # queries in two segments
    (100, 1090, 1090, 128, "fp16", None, True, 0.1, "1"),        # ... under a causal mask
    (40, 2100, 1300, 128, "bf16", None, True, 0.0, "0"),         # ... in three
]


@pytest.mark.parametrize("bh,sq,sk,d,dtype,mask,causal,p,pair", CASES)
def test_many_heads_give_the_bits_of_few(bh, sq, sk, d, dtype, mask, causal, p, pair, monkeypatch):
    q, k, v, do = (t.cuda() for t in make_qkv(bh, sq, sk, d, seed=sq + sk, std=0.7, dtype=dtype, with_dout=True))
    rows = bh // HPR
    m = lens = None
    if mask == "len":
        lens = torch.randint(0, sk + 1, (rows,), generator=torch.Generator().manual_seed(7), dtype=torch.int32)
        lens[1] = 0
        lens[-1] = sk
        lens = lens.cuda()
    elif mask:
        m = tail_mask(mask, rows, sk, seed=11).to(TDT[dtype]).cuda()
    kw = dict(causal=causal)
    if p > 0:
        kw.update(drop_kind=capi.DROP_PHILOX, p_drop=p, seed=99, offset=12)

    def args(h0, h1):
        r = slice(h0 // HPR, h1 // HPR)
        return dict(kw, mask=None if m is None else m[r], kv_len=None if lens is None else lens[r])

    try:
        if pair is not None:
            monkeypatch.setenv("FMHA_BWD_PAIR", pair)
            capi.lib().fmha_reload_overrides()
        o, lse, _, _ = capi.fwd(q, k, v, want_lse=True, **args(0, bh))
        fill = [torch.full_like(t, 7.0) for t in (q, k, v)]     # (every element has to be written)
        got = capi.bwd(do, q, k, v, o, lse, grads=fill, **args(0, bh))
        got = [t.clone() for t in got]
        again = capi.bwd(do, q, k, v, o, lse, **args(0, bh))
        torch.cuda.synchronize()
        for name, a, b in zip(("dq", "dk", "dv"), got, again):
            assert torch.equal(a, b), name
        # slices of two mask rows: the first, (without dropout: its decisions depend on the head's index) one inside, the last
        for h0 in (0,) if p > 0 else (0, rows // 2 * HPR, bh - 2 * HPR):
            h1 = h0 + 2 * HPR
            few = capi.bwd(do[h0:h1], q[h0:h1], k[h0:h1], v[h0:h1], o[h0:h1], lse[h0:h1].contiguous(), **args(h0, h1))
            torch.cuda.synchronize()
            for name, a, b in zip(("dq", "dk", "dv"), got, few):
                if causal and sq < 192:
                    b = b.float()
                    assert (a[h0:h1].float() - b).abs().max().item() <= 8 * U[dtype] * b.abs().max().item(), (name, h0)
                else:
                    assert torch.equal(a[h0:h1], b), (name, h0)
    finally:
        if pair is not None:
            monkeypatch.delenv("FMHA_BWD_PAIR")
            capi.lib().fmha_reload_overrides()
