"""Decode steps in pieces: the plan looks at sizes alone, so key counts give the bits of the mask that hides the same keys, and the workspace query may
be asked before the pointers are set."""
import ctypes as C
import pytest
import torch

from nvfuserexamples_amd import capi

pytestmark = pytest.mark.gpu

STEPS = [("fp16", 19, 2, 1708, 64), ("fp16", 33, 4, 1798, 64), ("fp16", 35, 2, 926, 128), ("fp16", 24, 2, 1299, 128), ("e4m3", 55, 3, 1057, 64),
         ("e4m3", 37, 2, 843, 128), ("e4m3", 8, 4, 12714, 128), ("fp16", 5, 1, 5000, 64)]


@pytest.mark.parametrize("kind,bh,sq,sk,d", STEPS)
def test_counts_are_the_mask(kind, bh, sq, sk, d):
    g = torch.Generator().manual_seed(sk)
    q, k, v = (torch.randn(bh, s, d, generator=g).half() for s in (sq, sk, sk))
    lens = torch.tensor([sk // 2 + int((i + 0.5) * (sk - sk // 2) / bh) for i in range(bh)], dtype=torch.int32)
    m = torch.where(torch.arange(sk)[None] < lens[:, None], 0.0, -10000.0).half().view(bh, 1, sk).cuda()
    if kind == "e4m3":
        f, t = capi.fwd_fp8, [x.to(torch.float8_e4m3fn).cuda() for x in (q, k, v)]
    else:
        f, t = capi.fwd, [x.cuda() for x in (q, k, v)]
    a, b = f(*t, mask=m, want_lse=True), f(*t, kv_len=lens.cuda(), want_lse=True)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


@pytest.mark.parametrize("kind,bh,sq,sk,d", STEPS)
def test_the_query_does_not_look_at_pointers(kind, bh, sq, sk, d):
    P, query = (capi.FwdFp8Params(), capi.lib().fmha_fwd_fp8_workspace_bytes) if kind == "e4m3" else (capi.FwdParams(), capi.lib().fmha_fwd_workspace_bytes)
    P.bh, P.sq, P.sk, P.d, P.scale = bh, sq, sk, d, d ** -0.5
    capi._sync_env()
    before = query(C.byref(P))
    P.kv_len, P.kv_len_bh_div = 4096, 1
    P.q = P.k = P.v = P.o = P.lse = 4096
    assert query(C.byref(P)) == before
