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


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,H,Nq,Nk,D", [(1, 4, 129, 1000, 64), (1, 3, 200, 777, 128), (2, 1, 257, 600, 256), (1, 40, 144, 300, 128),
                                         (1, 2, 512, 513, 64), (1, 2, 513, 514, 64)])
def test_long_blocks_on_the_short_kernel(qfa, B, H, Nq, Nk, D, causal):
    _check(qfa, B, H, Nq, Nk, D, causal, torch.float16, torch.float16, seed=Nq)


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
    q, o, code = q.detach(), o.detach(), {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}
    st = torch.cuda.current_stream().cuda_stream
    dense = lambda n: (H * n * D, n * D, D)
    ptr = lambda *ts: [t.data_ptr() for t in ts]

    o2, lse = torch.empty_like(q), torch.empty((B, H, Nq), device=DEV)
    ws = torch.empty(L.qfa_attn_fwd_cache_workspace_bytes(B, H, Nq, Nk, D), dtype=torch.uint8, device=DEV)
    assert L.qfa_attn_fwd_cache_lse(q.data_ptr(), code[dtype], *ptr(*kq, *vq), code[kq[1].dtype], *ptr(o2, lse), B, H, Nq, Nk, D,
                                    *dense(Nq), *dense(Nk), *dense(Nk), *dense(Nq), sm, 1, ws.data_ptr() if ws.numel() else None,
                                    ws.numel(), st) == 0, L.qfa_last_error()
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
                          ws.numel(), *ptr(*want), code[io], B, H, Nq, Nk, D, *dense(Nq), *dense(Nk), *dense(Nk), *dense(Nq),
                          *dense(Nq), *dense(Nq), *dense(Nk), *dense(Nk), sm, 1, st) == 0, L.qfa_last_error()
    for a, b in zip(grads, want):
        assert torch.equal(a, b.to(dtype))
