"""The decode kernel's banks (the four lanes that hold one score): every number of query rows, so that a bank holds a row or a key, with the last
keys of a block in any bank, keys hidden by the mask in some banks only, and e4m3 rows as fp16 over every value of the type."""
import numpy as np
import pytest
import torch

import oracle
from nvfuserexamples_amd import capi
from conftest import make_qkv, f32

pytestmark = pytest.mark.gpu

O_TOL = {"fp16": 2e-3, "bf16": 2e-2}       # as in test_gpu_decode.py


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("sq", [1, 2, 3, 4])
@pytest.mark.parametrize("sk,dtype", [(1, "fp16"), (5, "bf16"), (31, "fp16"), (33, "bf16"), (127, "fp16"), (130, "bf16"), (261, "fp16")])
def test_keys_and_rows_of_the_banks(sq, sk, d, dtype):
    bh = 6
    q, k, v = make_qkv(bh, sq, sk, d, seed=sk + sq, dtype=dtype)
    hidden = np.random.default_rng(sk).random((bh, 1, sk)) < 0.4
    hidden[:, :, sk // 2] = False
    hidden[1] = True                                    # all keys of a head, and every key but one
    hidden[2] = np.arange(sk)[None] != sk - 1
    m = torch.from_numpy(np.where(hidden, -np.inf, 0.25)).to(q.dtype)
    lens = torch.tensor([sk, sk, sk, 1, (sk + 1) // 2, 0], dtype=torch.int32)
    full = np.where(np.arange(sk)[None, None] < lens.numpy()[:, None, None], f32(m), -np.inf).astype(np.float32)
    full = np.broadcast_to(full, (bh, sq, sk)).copy()
    ref = oracle.attention(f32(q), f32(k), f32(v), mask=full, want=("o", "lse"))
    o, lse, _, _ = capi.fwd(q.cuda(), k.cuda(), v.cuda(), mask=m.cuda(), kv_len=lens.cuda(), want_lse=True)
    o, lse = f32(o.cpu()), lse.cpu().numpy()
    none = np.isneginf(full).all(-1)
    assert (o[none] == 0).all() and np.isneginf(lse[none]).all()
    assert np.abs(o[~none] - ref["o"][~none]).max() <= O_TOL[dtype]
    assert np.abs(lse[~none] - ref["lse"][~none]).max() <= 2e-3


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("sq", [1, 2, 4])
def test_every_e4m3_value(sq, d):
    """Keys that hold every finite byte once against queries of powers of two: products and sums are exact in fp32 (under 2^24 steps of
    2^-15), so the scores are, and the log-sum-exp is the float64 one's up to the fp32 exponentials and sum."""
    bytes_ = torch.tensor([b for b in range(256) if b & 0x7f != 0x7f], dtype=torch.uint8)
    sk = len(bytes_)
    k8 = torch.zeros(1, sk, d, dtype=torch.uint8)
    k8[0, torch.arange(sk), 7 * torch.arange(sk) % d] = bytes_
    k8 = k8.view(torch.float8_e4m3fn)
    q = torch.stack([2.0 ** -((torch.arange(d) + r) % 6) for r in range(sq)])[None]
    q8 = q.to(torch.float8_e4m3fn)
    assert torch.equal(q8.float(), q)
    v8 = torch.eye(sk, d)[None].to(torch.float8_e4m3fn)
    scale = 1.0 / 64
    _, lse = capi.fwd_fp8(q8.cuda(), k8.cuda(), v8.cuda(), scale=scale, want_lse=True)
    s = (q8.double() @ k8.double().transpose(1, 2)) * scale
    # 2^-24 per rounding: scale * log2(e) and the product 2, the exponent's argument (|s| <= 7, times log2(e)) and its exponential 4, the sum of 254 terms 8
    assert (lse.cpu().double() - torch.logsumexp(s, -1)).abs().max().item() <= 2.0 ** -24 * (7 * 1.5 * 4 + 4 + 16)
    nan = k8.clone().view(torch.uint8)
    nan[0, 3, 5] = 0x7f                                 # a NaN: what the same rows give in fp16
    nan = nan.view(torch.float8_e4m3fn)
    o, lse = capi.fwd_fp8(q8.cuda(), nan.cuda(), v8.cuda(), scale=scale, want_lse=True)
    o16, lse16, _, _ = capi.fwd(q8.half().cuda(), nan.half().cuda(), v8.half().cuda(), scale=scale, want_lse=True)
    assert torch.equal(o.isnan(), o16.isnan()) and torch.equal(lse.nan_to_num(), lse16.nan_to_num())
    assert not bool((lse.isfinite()).any())
