"""Shared-KV backward of query blocks that a workgroup holds: q, o and dO as the caller has them, cast and scaled inside, against the launches that cast
and scale first, and with gradients of very different size in different heads."""
import math

import pytest
import torch

from helpers import assert_close
from oracle import oracle
from quant_flash_attn_amd import _lib
from quant_flash_attn_amd.quant_flash_attn import _normalised_dout

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CODE = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}


def _tensors(B, H, Nq, Nk, D, dtype, sdtype):
    g = torch.Generator().manual_seed(Nq + Nk + D)
    r = lambda n: torch.randn((B, H, n, D), generator=g)
    q, o, do = (r(Nq).to(dtype).to(DEV) for _ in range(3))
    codes = torch.randint(-128, 128, (B, H, Nk, D), dtype=torch.int8, generator=g).to(DEV)
    scale = (torch.rand((B, H, Nk, 1), generator=g) * 0.02 + 0.001).to(sdtype).to(DEV)
    zp = torch.randint(-20, 20, (B, H, Nk, 1), dtype=torch.int8, generator=g).to(DEV)
    lse = (torch.rand((B, H, Nq), generator=g) * 2 + 6).to(DEV)
    return q, o, do, codes, scale, zp, lse


def _direct(q, o, do, codes, scale, zp, lse, sm, split):
    L = _lib.lib()
    B, H, Nq, D = q.shape
    Nk = codes.shape[2]
    dq, dkv = torch.empty_like(q), torch.empty((B, H, Nk, D), dtype=q.dtype, device=DEV)
    n = L.qfa_attn_bwd_shared_kv_workspace_bytes(B, H, Nq, Nk, D) if split else 0
    ws = torch.empty(max(n, 16), dtype=torch.uint8, device=DEV)
    st = lambda t: t.stride()[:3]
    rc = L.qfa_attn_bwd_shared_kv_direct(q.data_ptr(), codes.data_ptr(), scale.data_ptr(), CODE[scale.dtype], zp.data_ptr(),
                                         o.data_ptr(), do.data_ptr(), lse.data_ptr(), dq.data_ptr(), dkv.data_ptr(), CODE[q.dtype],
                                         CODE[do.dtype], CODE[q.dtype], B, H, Nq, Nk, D, *st(q), *st(codes), *st(o), *st(do), *st(dq),
                                         *st(dkv), sm, ws.data_ptr() if n else None, n, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, L.qfa_last_error()
    return dq, dkv, n


def _scaled_first(q, o, do, codes, scale, zp, lse, sm):
    do16, back = _normalised_dout(do, scale)
    return _lib.host().skv_bwd(q.half(), codes, scale, zp, o.half(), do16, lse, sm, q.dtype, back)


@pytest.mark.parametrize("dtype,sdtype", [(torch.float16, torch.float16), (torch.bfloat16, torch.float16), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("B,H,Nq,Nk,D", [(1, 1, 1, 33, 64), (1, 3, 16, 700, 128), (2, 3, 17, 257, 64), (1, 2, 32, 4000, 128),
                                         (1, 2, 5, 100, 256), (1, 4, 16, 3001, 256), (300, 2, 3, 31, 64),
                                         # two kernels: 16 or 32 queries per wave in dQ, keys split or not (1060 heads over 300 keys: one pass)
                                         (1, 4, 33, 700, 128), (20, 53, 97, 300, 128), (1, 2, 128, 4097, 64), (3, 64, 65, 1000, 64),
                                         (1, 1, 128, 31, 128), (20, 53, 97, 100, 128), (5, 56, 97, 300, 64),
                                         # one pass, a workgroup per head: ends of the scan for the largest key scale
                                         (2, 64, 40, 1024, 128), (4, 32, 97, 1025, 128), (1, 320, 40, 2049, 64), (5, 64, 97, 2048, 64)])
def test_direct_against_scaled_first(qfa, B, H, Nq, Nk, D, dtype, sdtype):
    t = _tensors(B, H, Nq, Nk, D, dtype, sdtype)
    t[2].mul_(1e-4)
    want = _scaled_first(*t, 0.09)
    for split in (False, True):
        got = _direct(*t, 0.09, split)
        for a, b in zip(got[:2], want):
            # another power of two per workgroup: the same products but for what binary16 loses below 2^-14 of the largest (2^-10
            # of such a value), and with a split another order of fp32 sums, rounded to 8 bits once
            assert (a.double() - b.double()).norm() <= 2.0 ** -8 * b.double().norm()
    assert _lib.lib().qfa_attn_bwd_shared_kv_is_direct(129, 64) == 0 and _lib.lib().qfa_attn_bwd_shared_kv_is_direct(17, 256) == 0


def test_heads_do_not_share_the_scaling(qfa):
    """Gradients 2^40 apart in two heads: each head's are as good as alone (one scaling for both loses the small ones)."""
    for Nq in (16, 100):
        _scaling_of_heads(Nq)


def _scaling_of_heads(Nq):
    q, o, do, codes, scale, zp, lse = _tensors(1, 2, Nq, 500, 128, torch.bfloat16, torch.float16)
    do[:, 0] *= 2.0 ** -40
    dq, dkv, _ = _direct(q, o, do, codes, scale, zp, lse, 0.09, False)
    for h in (0, 1):
        one = [x[:, h:h + 1].contiguous() for x in (q, o, do, codes, scale, zp, lse)]
        for a, b in zip((dq, dkv), _scaled_first(*one, 0.09)):
            # (up to 32 queries the same kernel and the same power of two)
            assert b.abs().max() > 0 and (a[:, h:h + 1].double() - b.double()).norm() <= (0 if Nq <= 32 else 2.0 ** -8) * b.double().norm()


@pytest.mark.parametrize("Nq", [7, 40, 100])
def test_infinite_and_zero_gradients(qfa, Nq):
    q, o, do, codes, scale, zp, lse = _tensors(1, 3, Nq, 100, 64, torch.float16, torch.float16)
    do[:, 0] = 0
    do[0, 1, 3, 5] = float("inf")
    dq, dkv, _ = _direct(q, o, do, codes, scale, zp, lse, 0.09, False)
    assert (dq[:, 0] == 0).all() and (dkv[:, 0] == 0).all()
    assert not torch.isfinite(dkv[:, 1]).all()
    assert torch.isfinite(dq[:, 2]).all() and torch.isfinite(dkv[:, 2]).all()


@pytest.mark.parametrize("dtype,sdtype", [(torch.float16, torch.float16), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("last", [False, True])
@pytest.mark.parametrize("Nq,Nk,D", [(16, 2048, 128), (32, 2048, 64), (16, 2048, 256),   # one pass, the keys split
                                     (64, 256, 128), (128, 2048, 128), (100, 3000, 64)])   # dKV by chunks of keys, dQ split or not
def test_small_keys_beside_large_ones(qfa, Nq, Nk, D, last, dtype, sdtype):
    """delta = rowsum(O o dO) holds every key of the head, a workgroup's own key scales do not: where its keys are 2^-6 beside
    others of 2^8 in the same head, dS = sm * p * (dP - delta) must stay within binary16 all the same."""
    g = torch.Generator().manual_seed(Nq + D)
    kv = torch.randn((1, 1, Nk, D), generator=g) * 2.0 ** -6
    half = slice(Nk // 2, None) if last else slice(0, Nk // 2)
    kv[:, :, half] = 256.0 * (1.0 + 64.0 * kv[:, :, half])
    q = (torch.randn((1, 1, Nq, D), generator=g) / 256.0).to(dtype)
    kv, do, sm = kv.to(dtype), torch.full((1, 1, Nq, D), 2.0 ** -6, dtype=dtype), 1.0 / math.sqrt(D)
    qd, kvd = q.to(DEV).requires_grad_(True), kv.to(DEV).requires_grad_(True)
    quant = qfa.asymmetric_quant_per_token(kvd.detach(), scale_dtype=sdtype)
    o = qfa.quant_flash_attn(qd, kvd, quant, sm)
    dq, dkv = torch.autograd.grad(o, [qd, kvd], do.to(DEV))
    (dq_ref, dkv_ref), (nq, nkv) = oracle.legacy_bwd(q, *(t.cpu() for t in quant), do, sm, o=o.detach().cpu(), spread=True)
    assert_close("dQ", dq.cpu(), dq_ref, scaled=True, spread=nq)
    for part in (slice(0, Nk // 2), slice(Nk // 2, None)):
        assert_close("dKV", dkv[:, :, part].cpu(), dkv_ref[:, :, part], scaled=True, spread=nkv[:, :, part])
