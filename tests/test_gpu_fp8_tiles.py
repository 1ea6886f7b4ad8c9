"""Key tiles of the e4m3 forward: those with and without a mask term, those left out behind the last live key of a mask
row, those past a wave's own causal rows.  Bounds against the oracle as in test_gpu_fp8.py; leaving tiles out must not
change a bit."""
import numpy as np
import pytest
import torch

import oracle
from nvfuserexamples_amd import capi
from conftest import f32

pytestmark = pytest.mark.gpu


def _inputs(bh, sq, sk, d, seed):
    g = torch.Generator().manual_seed(seed)
    out = []
    for s in (sq, sk, sk):
        x = torch.randn(bh, s, d, generator=g)
        f = float(x.abs().max()) / 448.0
        out += [(x / f).to(torch.float8_e4m3fn), f]
    return out


def _check(o, lse, q8, dq, k8, dk, v8, dv, d, mask, causal):
    qf, kf, vf = (f32(t.float()) for t in (q8, k8, v8))
    kw = dict(mask=mask, causal=causal, scale=d ** -0.5 * dq * dk, want=("o", "lse"))
    ref = oracle.attention(qf, kf, vf * np.float32(dv), round_p="e4m3", **kw)
    vmax, top = float(np.abs(vf).max()) * dv, np.abs(ref["o"]).max()
    dev = np.abs(f32(o.cpu()) - ref["o"])
    assert np.quantile(dev, 0.999) <= 2e-3 * vmax + 2.0 ** -11 * top
    assert dev.max() <= 2.0 ** -4 * vmax + 2.0 ** -11 * top
    assert np.abs(lse.cpu().numpy() - ref["lse"]).max() <= 2e-3


@pytest.mark.parametrize("d,sk", [(64, 65), (64, 512), (128, 300)])
@pytest.mark.parametrize("hidden", [-9000.0, -10000.0, float("-inf")])
def test_tiles_behind_the_last_live_key_are_left_out_exactly(d, sk, hidden, monkeypatch):
    lens = [1, 63, 64, sk - 1, sk, 0, sk // 2, sk // 2]  # (0: a row without a live key keeps all its keys)
    b, sq = len(lens), 70
    q8, dq, k8, dk, v8, dv = _inputs(b, sq, sk, d, sk)
    m = torch.zeros(b, 1, sk)
    for i, n in enumerate(lens):
        m[i, :, n:] = hidden if n or hidden > float("-inf") else -10000.0
    m[6, :, :5] = -10000.0              # hidden keys ahead of live ones
    m[7, :, : sk // 2] = -1500.0        # nothing at or above -1000: the row keeps its keys
    m = m.half()
    got = []
    for trim in ("1", "0"):
        monkeypatch.setenv("FMHA_MASK_TRIM", trim)
        capi.lib().fmha_reload_overrides()
        got.append(capi.fwd_fp8(q8.cuda(), k8.cuda(), v8.cuda(), dq, dk, dv, mask=m.cuda(), want_lse=True))
        torch.cuda.synchronize()
    monkeypatch.delenv("FMHA_MASK_TRIM")
    capi.lib().fmha_reload_overrides()
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    _check(*got[0], q8, dq, k8, dk, v8, dv, d, np.broadcast_to(f32(m), (b, sq, sk)).copy(), False)


def test_scores_that_could_reach_a_masked_key_keep_its_tile():
    """One query of value 448 against a hidden key of 448 at a scale of 0.001: its score, 12845, beats the mask."""
    q = torch.full((1, 8, 64), 448.0).to(torch.float8_e4m3fn)
    k = torch.zeros(1, 256, 64)
    k[:, 200] = 448.0
    v = torch.randn(1, 256, 64, generator=torch.Generator().manual_seed(0)).to(torch.float8_e4m3fn)
    m = torch.zeros(1, 1, 256)
    m[..., 100:] = -10000.0
    o, _ = capi.fwd_fp8(q.cuda(), k.to(torch.float8_e4m3fn).cuda(), v.cuda(), scale=0.001, mask=m.half().cuda())
    assert torch.equal(o.float().cpu(), v[:, 200:201].float().expand(1, 8, 64))


@pytest.mark.parametrize("bh,sq,sk,d", [(8, 33, 33, 64), (17, 200, 200, 64), (16, 130, 320, 64), (9, 320, 130, 128),
                                        (24, 1100, 1100, 64), (8, 129, 129, 128)])
def test_causal_tiles(bh, sq, sk, d):
    q8, dq, k8, dk, v8, dv = _inputs(bh, sq, sk, d, sq)
    o, lse = capi.fwd_fp8(q8.cuda(), k8.cuda(), v8.cuda(), dq, dk, dv, causal=True, want_lse=True)
    torch.cuda.synchronize()
    _check(o, lse, q8, dq, k8, dk, v8, dv, d, None, True)
