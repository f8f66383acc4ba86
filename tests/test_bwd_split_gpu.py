"""The backward with its streamed rows split over workgroups (few heads): dK and dV over the queries, dQ over the keys, against
fp64 and against the same kernels without the split."""
import math

import pytest
import torch

from helpers import assert_close
from oracle import oracle
from quant_flash_attn_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = [
    # B, H, Nq, Nk, D, causal, dtype
    (1, 2, 700, 700, 64, True, torch.bfloat16),
    (1, 1, 1001, 1001, 64, False, torch.float16),
    (2, 1, 333, 2100, 64, True, torch.float16),       # every query sees the first keys, few see the last part
    (1, 2, 1500, 1500, 128, True, torch.bfloat16),    # late keys are seen by the last part of the queries only
    (1, 3, 640, 900, 128, False, torch.float16),
    (1, 1, 2050, 2050, 128, True, torch.float32),     # two rows in the last block
    (1, 1, 65, 3000, 128, True, torch.bfloat16),
    (1, 2, 1100, 1100, 256, True, torch.bfloat16),
    (1, 2, 400, 1000, 256, True, torch.float16),
    (1, 1, 600, 530, 256, False, torch.float32),
]


def _inputs(B, H, Nq, Nk, D, dtype):
    g = torch.Generator().manual_seed(Nq + Nk + D)
    mk = lambda n: (torch.randn((B, H, n, D), generator=g) + 0.3 * torch.randn((B, H, n, 1), generator=g)).to(dtype).to(DEV)
    return mk(Nq), mk(Nk), mk(Nk), mk(Nq)


def _parts(B, H, Nq, Nk, D, causal):
    L = _lib.lib()
    return L.qfa_attn_bwd_split_workspace_bytes(B, H, Nq, Nk, D, int(causal), 0) - L.qfa_attn_bwd_workspace_bytes(B, H, Nq, Nk, D)


def _undivided(qq, kq, v, o, do, lse, causal, sm):
    """qfa_attn_bwd with the workspace that it has to have and no more"""
    L = _lib.lib()
    B, H, Nq, D = do.shape
    Nk = v.shape[2]
    ws = torch.empty(L.qfa_attn_bwd_workspace_bytes(B, H, Nq, Nk, D), dtype=torch.uint8, device=DEV)
    dq, dk, dv = torch.empty_like(do), torch.empty_like(v), torch.empty_like(v)
    dense = lambda n: (H * n * D, n * D, D)
    ptr = lambda *ts: [t.data_ptr() for t in ts]
    rc = L.qfa_attn_bwd(*ptr(qq.codes, qq.scale, qq.zero_point, qq.rowsum, kq.codes, kq.scale, kq.zero_point, kq.rowsum, v, o, do, lse, ws),
                        ws.numel(), *ptr(dq, dk, dv), {torch.float16: 1, torch.bfloat16: 2}[v.dtype], B, H, Nq, Nk, D, *dense(Nq),
                        *dense(Nk), *dense(Nk), *dense(Nq), *dense(Nq), *dense(Nq), *dense(Nk), *dense(Nk), sm, int(causal),
                        torch.cuda.current_stream().cuda_stream)
    assert rc == 0, L.qfa_last_error()
    return dq, dk, dv


@pytest.mark.parametrize("B,H,Nq,Nk,D,causal,dtype", CASES)
def test_split_backward(qfa, B, H, Nq, Nk, D, causal, dtype):
    assert _parts(B, H, Nq, Nk, D, causal) > 0, "the plan splits this shape"
    sm = 1.0 / math.sqrt(D)
    q, k, v, do = _inputs(B, H, Nq, Nk, D, dtype)
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    o = qfa.quant_flash_attn_qkv(*leaves, causal, sm)
    grads = torch.autograd.grad(o, leaves, do)
    q, k, v, o = (t.detach() for t in (q, k, v, o))
    io = torch.bfloat16 if dtype == torch.float32 else dtype
    v16, o16, do16 = (t.to(io) for t in (v, o, do))
    qq, kq = qfa.quantize_for_attention(q), qfa.quantize_for_attention(k)
    lse = qfa.attn_fwd_quantized(qq, kq, v16, causal, sm)[1]
    whole = _undivided(qq, kq, v16, o16, do16, lse, causal, sm)
    qh, kh = (oracle.dequantize_per_token(*(x.cpu() for x in t[:3]), torch.float64) for t in (qq, kq))
    refs, spreads = oracle.attn_bwd(qh, kh, v16.cpu(), do16.cpu(), causal, sm, o=o16.cpu(), spread=True)
    for name, got, un, want, sp in zip(("dQ", "dK", "dV"), grads, whole, refs, spreads):
        assert got.dtype == dtype
        assert_close(name, got.double().cpu(), want, scaled=True, rel=2.0 ** -7, spread=sp)
        # the same products of the same operands, added in another order and rounded once instead of never (2^-8 in bf16); the
        # two LSE differ by the rounding of the probabilities that they sum (2^-9)
        diff = (got.double() - un.double()).norm() / un.double().norm()
        assert diff < 2.0 ** -7, f"{name}: {float(diff)}"


def test_split_backward_keeps_infinities_apart(qfa):
    """An infinite dO row reaches the gradients of the keys that its query sees, in whatever part they are, and no others (dV:
    none behind its block of 32 queries, whose diagonal block multiplies the masked probabilities with it)."""
    B, H, N, D, sm, row = 1, 2, 1500, 128, 0.09, 700
    assert _parts(B, H, N, N, D, True) > 0
    q, k, v, do = _inputs(B, H, N, N, D, torch.bfloat16)
    do[:, :, row] = math.inf
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    dq, dk, dv = torch.autograd.grad(qfa.quant_flash_attn_qkv(*leaves, True, sm), leaves, do)
    keep = torch.arange(N, device=DEV) != row
    assert torch.isfinite(dq[:, :, keep]).all()
    assert torch.isfinite(dk[:, :, row + 1:]).all()
    assert torch.isfinite(dv[:, :, row // 32 * 32 + 32:]).all()
    assert not torch.isfinite(dv[:, :, :row + 1]).any()


def test_split_backward_replayed_from_a_graph(qfa):
    B, H, N, D, sm = 1, 2, 1024, 128, 0.09
    assert _parts(B, H, N, N, D, True) > 0
    q, k, v, do = _inputs(B, H, N, N, D, torch.bfloat16)
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    step = lambda: torch.autograd.grad(qfa.quant_flash_attn_qkv(*leaves, True, sm), leaves, do)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = step()
    for _ in range(3):
        graph.replay()
        want = step()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        do.neg_()
