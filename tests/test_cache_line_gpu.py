"""Query blocks of more than 128 on an INT8 cache that take the short-query kernel because its few launches win there: ragged last
blocks of 16, the last length that may take it and the first that may not, against fp64."""
import math

import pytest
import torch

from helpers import max_abs
from oracle import oracle
from quant_flash_attn_amd import _lib
from quant_flash_attn_amd.synthetic import make_inputs
from test_cache_gpu import _check

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


CODE = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}
_ptr = lambda *ts: [t.data_ptr() for t in ts]
_dense = lambda H, n, D: (H * n * D, n * D, D)


def _short_kernel(q, kq, vq, causal, sm):
    """O and LSE of qfa_attn_fwd_cache_lse, dense tensors"""
    L = _lib.lib()
    B, H, Nq, D = q.shape
    Nk = kq[0].shape[2]
    o, lse = torch.empty_like(q), torch.empty((B, H, Nq), device=DEV)
    ws = torch.empty(L.qfa_attn_fwd_cache_workspace_bytes(B, H, Nq, Nk, D), dtype=torch.uint8, device=DEV)
    strides = [s for n in (Nq, Nk, Nk, Nq) for s in _dense(H, n, D)]
    assert L.qfa_attn_fwd_cache_lse(q.data_ptr(), CODE[q.dtype], *_ptr(*kq, *vq), CODE[kq[1].dtype], *_ptr(o, lse), B, H, Nq, Nk, D,
                                    *strides, sm, int(causal), ws.data_ptr() if ws.numel() else None, ws.numel(),
                                    torch.cuda.current_stream().cuda_stream) == 0, L.qfa_last_error()
    return o, lse


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,H,Nq,Nk,D,short", [(1, 4, 129, 1000, 64, True), (1, 3, 200, 777, 128, True), (2, 1, 257, 600, 256, True),
                                               (1, 40, 144, 300, 128, True), (1, 2, 512, 513, 64, True), (1, 2, 513, 514, 64, False),
                                               (8, 8, 333, 1500, 128, False)])
def test_long_blocks_on_the_short_kernel(qfa, B, H, Nq, Nk, D, short, causal):
    _check(qfa, B, H, Nq, Nk, D, causal, torch.float16, torch.float16, seed=Nq)
    # which of the two took the call: the other one rounds V, and its probabilities, in other places
    sm = 1.0 / math.sqrt(D)
    q, k, v, _ = (t.to(DEV) for t in make_inputs("offset", B, H, Nk, D, seed=Nq, dtype=torch.float16))
    q, kq, vq = q[:, :, :Nq].contiguous(), qfa.asymmetric_quant_per_token(k), qfa.asymmetric_quant_per_token(v)
    none = torch.empty(0, dtype=torch.float16, device=DEV)
    o = qfa.quant_flash_attn_quantized_kv(q, none, none, kq, vq, causal, sm)
    assert torch.equal(o, _short_kernel(q, kq, vq, causal, sm)[0]) == short


@pytest.mark.parametrize("B,H,Nq,Nk,D", [(1, 4, 129, 1000, 64), (1, 3, 200, 777, 128), (2, 1, 257, 600, 256), (1, 2, 512, 9001, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_gradient_of_the_short_kernels_output(qfa, B, H, Nq, Nk, D, dtype):
    """A call that wants a gradient runs one forward there: its O and LSE (against fp64) are what the backward takes."""
    L, sm, io = _lib.lib(), 1.0 / math.sqrt(D), torch.bfloat16 if dtype == torch.float32 else dtype
    q, k, v, do = (t.to(DEV) for t in make_inputs("offset", B, H, Nk, D, seed=Nq, dtype=dtype))
    q, do = q[:, :, :Nq].contiguous(), do[:, :, :Nq].contiguous()
    kq, vq = (qfa.asymmetric_quant_per_token(t) for t in (k, v))
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    o = qfa.quant_flash_attn_quantized_kv(*leaves, kq, vq, True, sm)
    grads = torch.autograd.grad(o, leaves, do)
    q, o = q.detach(), o.detach()
    dense, ptr = lambda n: _dense(H, n, D), _ptr

    o2, lse = _short_kernel(q, kq, vq, True, sm)
    assert torch.equal(o, o2)
    qq = qfa.quantize_for_attention(q)
    qh, kh = (oracle.dequantize_per_token(*(x.cpu() for x in t[:3]), torch.float64) for t in (qq, kq))
    vh = oracle.dequantize_per_token(*(t.cpu() for t in vq), torch.float64)
    # scores of order ten: binary32 rounds them and their exponentials to 2^-23 of that, a few times
    assert max_abs(lse.cpu(), oracle.attn_fwd(qh, kh, vh, True, sm)[1]) < 2.0 ** -16

    v16, do16, o16 = _lib.host().dequant(*vq, io), do.to(io), o.to(io)
    kr = kq[0].sum(-1, dtype=torch.int32)
    ws = torch.empty(L.qfa_attn_bwd_split_workspace_bytes(B, H, Nq, Nk, D, 1, 0), dtype=torch.uint8, device=DEV)
    want = torch.empty_like(do16), torch.empty_like(v16), torch.empty_like(v16)
    assert L.qfa_attn_bwd(*ptr(qq.codes, qq.scale, qq.zero_point, qq.rowsum, kq[0], kq[1].float(), kq[2], kr, v16, o16, do16, lse, ws),
                          ws.numel(), *ptr(*want), CODE[io], B, H, Nq, Nk, D, *dense(Nq), *dense(Nk), *dense(Nk), *dense(Nq),
                          *dense(Nq), *dense(Nq), *dense(Nk), *dense(Nk), sm, 1,
                          torch.cuda.current_stream().cuda_stream) == 0, L.qfa_last_error()
    for a, b in zip(grads, want):
        assert torch.equal(a, b.to(dtype))
