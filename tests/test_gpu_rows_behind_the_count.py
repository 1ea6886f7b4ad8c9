"""K and V rows at and past a head's key count hold anything (a cache from an uninitialised allocation): the forward gives the bits that finite
rows give.  The kernel whose waves share 32 queries with one, four and eight waves and in pieces, and every other forward that takes counts; on both
sides of the kernels' blocks of 32 and 64 keys, with an additive mask and the causal mask beside the counts, folded and packed rows, a count of none and of all
keys (without any, the other forwards go through the head's first row with weights of zero: that one is finite)."""
import pytest
import torch

from nvfuserexamples_amd import capi

pytestmark = pytest.mark.gpu


def _bits(sq, sk, d, dtype=torch.float16, causal=False, mask=False, packed=False, h=2, flags=4, first=0, **kw):
    b = 7
    g = torch.Generator().manual_seed(sk + d)
    lens = torch.tensor([0, 1, sk // 3, min(sk, 33), (sk // 64) * 64 or 1, sk - 1, sk], dtype=torch.int32)
    q = torch.randn(b, h, sq, d, generator=g).to(dtype) * 0.5
    kv = torch.randn(b, sk, 2, h, d, generator=g).to(dtype) * 0.5
    m = (torch.randn(b, 1, 1, sk, generator=g) * 0.5).to(dtype).cuda() if mask else None
    got = []
    for fill in (None, float("nan"), float("inf")):
        x = kv.clone()
        if fill is not None:
            x[torch.arange(sk)[None] >= lens[:, None].clamp_min(first)] = fill
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


@pytest.mark.parametrize("sq,sk,d,causal,mask,packed,kw", [
    (100, 100, 64, False, False, False, {}), (128, 128, 64, False, True, True, {}), (40, 60, 64, False, False, False, dict(drop_kind=1, p_drop=0.1)),   # one pass
    (200, 200, 64, False, True, False, {}), (197, 197, 64, False, False, True, {}), (256, 256, 64, True, True, False, {}),                            # K and V in LDS
    (512, 400, 64, False, True, False, dict(h=64)), (512, 512, 64, False, False, True, dict(h=64)),                                                    # whole head
    (300, 700, 64, False, False, False, {}), (300, 300, 128, True, False, True, {}), (200, 333, 96, False, True, True, {}),                            # pipelined
    (1024, 1100, 64, False, False, False, dict(h=64)),                                                                                                 # .. two blocks a wave
    (50, 60, 256, False, False, False, {}), (200, 300, 256, False, True, False, {}),                                                                   # head dim 256
    (1, 300, 64, False, False, False, {}), (3, 700, 128, False, True, True, {}),                                                                       # decode steps
])
def test_the_other_kernels(sq, sk, d, causal, mask, packed, kw, monkeypatch):
    monkeypatch.setenv("FMHA_FWD_FEW", "0")
    _bits(sq, sk, d, torch.float16, causal, mask, packed, flags=0, workspace=False, first=1, **kw)


@pytest.mark.parametrize("sq,sk,d", [(2, 700, 64), (9, 700, 64), (40, 640, 128), (30, 500, 256)])
def test_their_pieces(sq, sk, d, monkeypatch):
    monkeypatch.setenv("FMHA_FWD_SPLIT", "3")
    _bits(sq, sk, d, mask=True, flags=0, first=1)
