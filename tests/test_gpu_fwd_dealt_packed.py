"""Causal forwards of packed bf16 rows with dropout at head dim 128 whose items are dealt by length: full and ragged last tiles, the
whole width and narrower rows, against the same rows folded (another kernel)."""
import pytest
import torch

from nvfuserexamples_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,h,s,d", [(3, 8, 1800, 128), (3, 8, 1792, 128), (2, 12, 1345, 128), (5, 8, 1100, 112)])
def test_dealt_packed_rows_give_what_folded_rows_give(b, h, s, d):
    g = torch.Generator().manual_seed(s + d)
    qkv = torch.randn(b, s, 3, h, d, generator=g).bfloat16().cuda()
    packed = [qkv[:, :, i].transpose(1, 2) for i in range(3)]
    folded = [t.reshape(b * h, s, d).contiguous() for t in packed]
    kw = dict(causal=True, drop_kind=capi.DROP_PHILOX, p_drop=0.1, seed=5, offset=9, want_lse=True)
    o, lse, _, _ = capi.fwd(*packed, **kw)
    o2, lse2, _, _ = capi.fwd(*folded, **kw)
    torch.cuda.synchronize()
    a, c = o.reshape(b * h, s, d).float().cpu(), o2.float().cpu()
    # The two round the same probabilities and outputs, but may take another reference exponent: half a unit for each of the four, row
    # by row, so that the keys of the last tile count: the last row's output without them is off by sqrt(8 / 1800), 1 / sqrt(1345) and
    # sqrt(12 / 1100) of its size.
    assert ((a - c).norm(dim=-1) <= 2 * 2.0 ** -8 * c.norm(dim=-1)).all()
    assert torch.allclose(lse.reshape(b * h, s).cpu(), lse2.cpu(), rtol=0, atol=2.0 ** -8)
