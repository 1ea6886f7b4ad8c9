"""A query row's result on e4m3 inputs is its own, to the bit, whatever rows share its wave: rows that raise their reference again and again (and whose
probabilities overflow e4m3 before they do), or hold NaN, in one half of every 32 rows, and the other half beside ordinary ones."""
import pytest
import torch

from nvfuserexamples_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["0", "1"])
@pytest.mark.parametrize("sq,sk,d,causal,masked", [(64, 700, 64, False, False), (100, 520, 64, True, False), (33, 700, 64, False, True), (70, 600, 128, False, True),
                                                   (64, 900, 128, True, False)])
def test_rows_apart(sq, sk, d, causal, masked, form, monkeypatch):
    monkeypatch.setenv("FMHA_FP8_SPLIT", form)
    b = 4
    g = torch.Generator().manual_seed(sk)
    q, k, v = (torch.randn(b, s, d, generator=g) * 2 for s in (sq, sk, sk))
    k[:, ::97] *= 3                                    # (keys that lift a row's maximum well behind its first tile)
    m = None
    if masked:
        m = torch.where(torch.arange(sk)[None] < torch.tensor([sk, sk - 1, sk // 2, 3])[:, None], 0.0, -10000.0).half().view(b, 1, sk).cuda()
    k8, v8 = (x.to(torch.float8_e4m3fn).cuda() for x in (k, v))

    def run(x):
        return capi.fwd_fp8(x.to(torch.float8_e4m3fn).cuda(), k8, v8, mask=m, causal=causal, want_lse=True)

    o, lse = run(q)
    assert torch.isfinite(o).all()
    half = torch.arange(sq) % 32 // 16
    for other in (0, 1):
        for factor in (16.0, float("nan")):
            x = q.clone()
            x[:, half == other] *= factor
            o1, lse1 = run(x)
            same = (half != other).cuda()
            assert torch.equal(o1[:, same], o[:, same]) and torch.equal(lse1[:, same], lse[:, same]), (other, factor)
            assert bool(torch.isnan(o1[:, ~same]).all()) == (factor != factor)
