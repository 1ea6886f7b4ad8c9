"""K and V rows at and past a head's key count hold anything (a cache from an uninitialised allocation): the forward gives the bits that finite
rows give.  The kernel whose waves share 32 queries with one, four and eight waves and in pieces, on both sides of its blocks of 32 and 64 keys, with
an additive mask and the causal mask beside the counts, folded and packed rows, a count of none and of all keys."""
import pytest
import torch

from nvfuserexamples_amd import capi

pytestmark = pytest.mark.gpu


def _bits(sq, sk, d, dtype=torch.float16, causal=False, mask=False, packed=False, b=7, h=2, flags=4, **kw):
    g = torch.Generator().manual_seed(sk + d)
    lens = torch.tensor([0, 1, sk // 3, min(sk, 33), (sk // 64) * 64 or 1, sk - 1, sk], dtype=torch.int32)
    q = torch.randn(b, h, sq, d, generator=g).to(dtype) * 0.5
    kv = torch.randn(b, sk, 2, h, d, generator=g).to(dtype) * 0.5
    m = (torch.randn(b, 1, 1, sk, generator=g) * 0.5).to(dtype).cuda() if mask else None
    got = []
    for fill in (None, float("nan"), float("inf")):
        x = kv.clone()
        if fill is not None:
            x[torch.arange(sk)[None] >= lens[:, None]] = fill
        k, v = (x.cuda()[:, :, i].transpose(1, 2) for i in (0, 1))
        t = [q.cuda(), k, v] if packed else [t.reshape(b * h, -1, d).contiguous() for t in (q.cuda(), k, v)]
        o, lse, _, _ = capi.fwd(*t, mask=m, kv_len=lens.cuda(), causal=causal, want_lse=True, flags=flags, **kw)
        got.append((o, lse))
    o, lse = got[0]
    assert torch.isfinite(o).all() and not o.reshape(b, h, sq, d)[0].any()
    for o1, lse1 in got[1:]:
        assert torch.equal(o1, o) and torch.equal(lse1, lse)


@pytest.mark.parametrize("waves", ["1", "4", "8"])
@pytest.mark.parametrize("sq,sk,d,dtype,causal,mask,packed", [
    (5, 100, 64, torch.float16, False, False, False), (40, 600, 64, torch.bfloat16, False, True, False), (70, 150, 64, torch.float16, True, False, True),
    (33, 90, 128, torch.float16, False, False, False), (9, 300, 128, torch.bfloat16, False, True, True), (20, 70, 32, torch.float16, False, False, True),
    (64, 200, 96, torch.float16, True, True, False), (30, 130, 80, torch.float16, False, False, True), (33, 140, 256, torch.float16, False, False, False),
])
def test_shared_queries(sq, sk, d, dtype, causal, mask, packed, waves, monkeypatch):
    monkeypatch.setenv("FMHA_FWD_FEW", waves)
    _bits(sq, sk, d, dtype, causal, mask, packed, workspace=False)


@pytest.mark.parametrize("sq,sk,d,mask,packed", [(9, 700, 64, False, False), (40, 900, 128, True, True), (5, 640, 256, False, False), (17, 500, 96, True, False)])
def test_pieces(sq, sk, d, mask, packed, monkeypatch):
    monkeypatch.setenv("FMHA_FWD_SPLIT", "3")
    _bits(sq, sk, d, mask=mask, packed=packed)
