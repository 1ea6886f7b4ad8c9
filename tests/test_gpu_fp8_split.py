"""The e4m3 forward whose four waves take the key tiles of 32 queries in turn: waves without a tile, with one, with tiles the
end of the keys / the diagonal / the masks pass through, rows whose keys are all hidden in some waves' tiles.  Against
the oracle with the same rounding (bounds as in test_gpu_fp8_tiles.py) and against the form without the split."""
import numpy as np
import pytest
import torch

from nvfuserexamples_amd import capi, load_ops
from conftest import f32
from test_gpu_fp8_tiles import _check, _inputs

pytestmark = pytest.mark.gpu


def _both(monkeypatch, *args, **kw):
    got = []
    for split in ("1", "0"):
        monkeypatch.setenv("FMHA_FP8_SPLIT", split)
        got.append(capi.fwd_fp8(*args, want_lse=True, **kw))
        torch.cuda.synchronize()
    monkeypatch.delenv("FMHA_FP8_SPLIT")
    return got


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("sq,sk,causal", [(1, 1, False), (5, 64, False), (33, 65, False), (32, 256, False), (31, 257, True),
                                          (70, 193, True), (200, 300, False), (129, 577, True), (40, 1100, False), (300, 40, True)])
def test_waves_that_split_the_keys(sq, sk, causal, d, monkeypatch):
    monkeypatch.setenv("FMHA_FWD_DECODE", "0")
    bh = 3
    q8, dq, k8, dk, v8, dv = _inputs(bh, sq, sk, d, sq + sk)
    (o, lse), (o0, lse0) = _both(monkeypatch, q8.cuda(), k8.cuda(), v8.cuda(), dq, dk, dv, causal=causal)
    monkeypatch.delenv("FMHA_FWD_DECODE")
    _check(o, lse, q8, dq, k8, dk, v8, dv, d, None, causal)
    # Partial sums of up to 1 100 fp32 terms in another order (2^-24 sqrt(n) each way, under 1e-5 relative); where a wave's reference lies below the row's,
    # probabilities that rounded to 2^-9 steps there keep their three mantissa bits: half a step of a weight under 2^-6.
    vmax = float(v8.float().abs().max()) * dv
    assert (o.float() - o0.float()).abs().max().item() <= 2.0 ** -10 * vmax + 2.0 ** -10 * o0.float().abs().max().item()
    assert (lse - lse0).abs().max().item() <= 1e-5 * max(1.0, lse0.abs().max().item())


@pytest.mark.parametrize("d,sk", [(64, 300), (128, 577)])
def test_masked_tiles_of_some_waves(d, sk, monkeypatch):
    """Rows whose live keys lie in one wave's tiles only, at the start or the end, under -inf and -10000, and rows without any."""
    spans = [(0, 1), (0, 64), (64, 65), (128, 200), (sk - 1, sk), (sk - 70, sk), (0, sk), (0, 0)]
    b, sq = len(spans), 45
    q8, dq, k8, dk, v8, dv = _inputs(b, sq, sk, d, sk)
    for hidden in (-10000.0, float("-inf")):
        m = torch.full((b, 1, sk), hidden)
        for i, (lo, hi) in enumerate(spans):
            m[i, :, lo:hi] = 0.0
        m = m.half()
        (o, lse), (o0, lse0) = _both(monkeypatch, q8.cuda(), k8.cuda(), v8.cuda(), dq, dk, dv, mask=m.cuda())
        n = b if hidden > float("-inf") else b - 1      # (a row hidden by -inf throughout: zeros and -inf, below)
        _check(o[:n], lse[:n], q8[:n], dq, k8[:n], dk, v8[:n], dv, d, np.broadcast_to(f32(m[:n]), (n, sq, sk)).copy(), False)
        if n < b:
            assert torch.equal(o[n:], torch.zeros_like(o[n:])) and bool(torch.isneginf(lse[n:]).all())
            assert torch.equal(o0[n:], o[n:]) and torch.equal(lse0[n:], lse[n:])


@pytest.mark.parametrize("sq,sk,d,causal", [(300, 600, 64, False), (600, 600, 64, True), (257, 700, 128, False), (700, 1100, 128, True)])
def test_the_flag_decides(sq, sk, d, causal, monkeypatch):
    """Without FMHA_FLAG_SPLIT_KEYS a head's bits are those it has in a launch of many heads; with it, as from the operator, few heads take the split
    form."""
    b, few = 200, 3
    g = torch.Generator(device="cuda").manual_seed(sk)
    q8, k8, v8 = (torch.randn(b, s, d, device="cuda", generator=g).to(torch.float8_e4m3fn) for s in (sq, sk, sk))
    head = [x[:few].contiguous() for x in (q8, k8, v8)]
    o, lse = capi.fwd_fp8(q8, k8, v8, causal=causal, want_lse=True)
    o1, lse1 = capi.fwd_fp8(*head, causal=causal, want_lse=True)
    assert torch.equal(o1, o[:few]) and torch.equal(lse1, lse[:few])
    flagged = capi.fwd_fp8(*head, causal=causal, want_lse=True, flags=capi.FLAG_SPLIT_KEYS)
    op = load_ops().fmha_fwd_fp8(*head, 1.0, 1.0, 1.0, None, 0.0, causal)
    split, whole = _both(monkeypatch, *head, causal=causal)
    assert not torch.equal(split[0], whole[0])
    for got in (flagged, op):
        assert torch.equal(got[0], split[0]) and torch.equal(got[1], split[1])
    assert torch.equal(o1, whole[0]) and torch.equal(lse1, whole[1])
