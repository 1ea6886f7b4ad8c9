"""The saving forward's builds for few key tiles (two waves per SIMD): up to 192 keys at head dim 64, 64 at 128, and 128 there where
workgroups outnumber the compute units; O is that of the plain forward."""
import pytest
import torch

from oracle import eager
from nvfuserexamples_amd import capi

pytestmark = pytest.mark.gpu

TDT = {"fp16": torch.float16, "bf16": torch.bfloat16}
TOL = {"fp16": (2e-3, 1e-3), "bf16": (1.6e-2, 8e-3)}   # context, saved outputs, as in test_gpu_rows.py


@pytest.mark.parametrize("bh,sq,sk,d,dtype", [
    (3, 130, 129, 64, "fp16"), (3, 40, 191, 64, "bf16"), (3, 129, 192, 64, "fp16"), (3, 33, 193, 64, "fp16"),
    (3, 40, 8, 128, "fp16"), (3, 129, 63, 128, "bf16"), (3, 64, 64, 128, "fp16"), (3, 40, 65, 128, "fp16"),
    (257, 20, 65, 128, "fp16"), (257, 33, 127, 128, "bf16"), (300, 20, 128, 128, "fp16"), (257, 20, 129, 128, "fp16"),
])
def test_saved_outputs(bh, sq, sk, d, dtype):
    g = torch.Generator(device="cuda").manual_seed(sk + d)
    q, k, v = (torch.randn((bh, s, d), dtype=TDT[dtype], device="cuda", generator=g) for s in (sq, sk, sk))
    m1, m2 = (torch.randint(0, 2, (bh, sq, sk), device="cuda", generator=g).to(TDT[dtype]) for _ in range(2))
    m1[:, :, 0] = 1
    pad = (1 - m1) * -1000
    kw = dict(mask=pad, drop_kind=capi.DROP_TENSOR, drop_mask=m2, drop_scale=2.0)
    plain = capi.fwd(q, k, v, **kw)[0]
    o, _, sm, dr = capi.fwd(q, k, v, save=True, **kw)
    assert torch.equal(o, plain)
    want_sm, want_dr, ctx = eager.train_mha(q, k, v, pad, m2, keep_prob=0.5)
    to, ts = TOL[dtype]
    for got, want, tol in ((o, ctx, to), (sm, want_sm, ts), (dr, want_dr, 2 * ts)):
        assert (got.float() - want.float()).abs().max().item() <= tol * max(1.0, want.float().abs().max().item())
