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
