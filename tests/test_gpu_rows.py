"""The reference's operators (fmha/fmha_manual.cpp:39-47, 891-897) away from rows of whole 16-byte pieces and from head
dim 64: key counts around the tiles of the kernels that move [.., sq, sk] tensors as whole rows, against the same
composition in fp32."""
import pytest
import torch

from oracle import eager
from nvfuserexamples_amd import capi

pytestmark = pytest.mark.gpu

TDT = {"fp16": torch.float16, "bf16": torch.bfloat16}
TOL = {"fp16": (2e-3, 1e-3), "bf16": (1.6e-2, 8e-3)}   # context, saved outputs


def _inputs(bh, sq, sk, d, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    q, k, v = (torch.randn((bh, s, d), dtype=TDT[dtype], device="cuda", generator=g) for s in (sq, sk, sk))
    m1, m2 = (torch.randint(0, 2, (bh, sq, sk), device="cuda", generator=g).to(TDT[dtype]) for _ in range(2))
    m1[:, :, 0] = 1          # (a row with no visible key is not what these cases are about)
    return q, k, v, m1, m2


def _close(a, b, tol):
    assert (a.float() - b.float()).abs().max().item() <= tol * max(1.0, b.float().abs().max().item())


@pytest.mark.parametrize("sq,sk,d,dtype", [
    (33, 8, 64, "fp16"), (130, 9, 64, "fp16"), (64, 63, 64, "bf16"), (31, 127, 64, "fp16"), (128, 121, 64, "fp16"),
    (40, 129, 64, "fp16"), (200, 222, 64, "bf16"), (129, 511, 64, "fp16"), (64, 513, 64, "fp16"), (50, 582, 64, "fp16"),
    (33, 8, 128, "fp16"), (70, 63, 128, "bf16"), (128, 128, 128, "fp16"), (130, 190, 128, "fp16"), (40, 512, 128, "fp16"),
    (129, 517, 128, "fp16"), (64, 640, 128, "bf16"),
])
def test_operators_on_rows_of_any_length(sq, sk, d, dtype):
    import mha_manual  # noqa: F401
    ops = torch.ops.mha_manual
    q, k, v, m1, m2 = _inputs(3, sq, sk, d, dtype, seed=sk + d)
    to, ts = TOL[dtype]
    _close(ops.fmha_nvfuser(q, k, v, m1), eager.infer_mha(q, k, v, m1), to)
    pad = (1 - m1) * -1000
    sm, dr, ctx = eager.train_mha(q, k, v, pad, m2, keep_prob=0.5)
    plain = ops.fmha_train_nvfuser(q, k, v, pad, m2)
    saved = ops.fmha_train_saveim_nvfuser(q, k, v, pad, m2)
    _close(plain, ctx, to)
    assert torch.equal(saved[0], plain)
    _close(saved[1], sm, ts)
    _close(saved[2], dr, 2 * ts)


@pytest.mark.parametrize("sk,d", [(100, 64), (205, 64), (205, 128)])
def test_mask_rows_that_start_anywhere(sk, d):
    """A mask tensor with a pitch and a first element off every 16-byte boundary, read where it is."""
    q, k, v, m1, _ = _inputs(2, 70, sk, d, "fp16", seed=7)
    flat = torch.zeros(2 * 70 * sk + 3, dtype=torch.float16, device="cuda")
    mask = flat[3:].view(2, 70, sk)
    mask.copy_((1 - m1) * -1000)
    o = capi.fwd(q, k, v, mask=mask)[0]
    _close(o, eager.general_mha(q, k, v, mask), 2e-3)
