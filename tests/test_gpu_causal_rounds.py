"""Causal forwards of more (head, query tile) items than the persistent grid has workgroups, with tile counts that do not
divide the grid: some heads then lie in two rounds, and every one of their rows must still be computed."""
import pytest
import torch

from nvfuserexamples_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("s", [300, 768, 1200])
@pytest.mark.parametrize("d,dtype,p", [(64, torch.float16, 0.0), (64, torch.bfloat16, 0.1), (128, torch.bfloat16, 0.0), (96, torch.float16, 0.1)])
def test_heads_in_two_rounds_are_computed_whole(s, d, dtype, p):
    bh = 3 * 1024 // ((s + 127) // 128) + 1  # three rounds and a bit at two workgroups per compute unit
    g = torch.Generator(device="cuda").manual_seed(s + d)
    q, k, v = (torch.randn(bh, s, d, dtype=dtype, device="cuda", generator=g) for _ in range(3))
    kw = dict(causal=True, want_lse=True)
    o, lse, _, _ = capi.fwd(q, k, v, **kw)
    if p > 0:  # the dropout build: what a row keeps depends on its head, so against itself without dropout only the LSE
        lse_d = capi.fwd(q, k, v, drop_kind=capi.DROP_PHILOX, p_drop=p, seed=5, offset=1, **kw)[1]
        assert torch.equal(lse, lse_d)
    for i in range(0, bh, 40):   # few heads at a time: one round
        oi, li, _, _ = capi.fwd(q[i:i + 40], k[i:i + 40], v[i:i + 40], **kw)
        assert torch.equal(o[i:i + 40], oi) and torch.equal(lse[i:i + 40], li)


@pytest.mark.parametrize("bh,s,d,dtype,p,lens,packed", [
    (17, 2100, 64, torch.float16, 0.0, False, False),     # less than a round, one group of heads
    (34, 2100, 64, torch.bfloat16, 0.1, False, False),    # a round and a bit, two groups
    (44, 2500, 128, torch.bfloat16, 0.0, False, True),    # two rounds, four groups; run-time rows
    (104, 1500, 128, torch.float16, 0.0, True, False),    # two and a half, eight groups; key counts, among them 0
    (300, 520, 64, torch.bfloat16, 0.0, False, False),    # three
    (12, 3000, 256, torch.float16, 0.0, False, False),    # one workgroup per compute unit
    (40, 1000, 96, torch.float16, 0.1, False, True),
])
def test_items_dealt_by_length_are_computed_whole(bh, s, d, dtype, p, lens, packed):
    """Half a round to four rounds of causal items: dealt by length.  Every head as in a launch of its own, to the bit (the
    arithmetic does not depend on the dealing; with dropout, where it depends on a head's number, the LSE, which does not)."""
    g = torch.Generator(device="cuda").manual_seed(s + d)
    q, k, v = (torch.randn(bh, s, d, dtype=dtype, device="cuda", generator=g) for _ in range(3))
    n = None
    if lens:
        n = torch.randint(0, s + 1, (bh,), generator=torch.Generator().manual_seed(3), dtype=torch.int32)
        n[0] = 0
        n = n.cuda()
    kw = dict(causal=True, want_lse=True)
    if p > 0:
        kw.update(drop_kind=capi.DROP_PHILOX, p_drop=p, seed=5, offset=1)
    ins = [q, k, v]
    if packed:
        ins = [t.view(bh // 4, 4, s, d).transpose(1, 2).contiguous().transpose(1, 2) for t in ins]
    o, lse, _, _ = capi.fwd(*ins, kv_len=n, **kw)
    o, lse = o.reshape(bh, s, d), lse.reshape(bh, s)
    assert torch.isfinite(o.float()).all()
    for i in range(bh):
        oi, li, _, _ = capi.fwd(q[i:i + 1], k[i:i + 1], v[i:i + 1], workspace=False, kv_len=None if n is None else n[i:i + 1], **kw)
        assert torch.equal(lse[i], li.reshape(s)), i
        if p == 0 or i == 0:
            assert torch.equal(o[i], oi.reshape(s, d)), i
