"""fp32 tensors through quant_flash_attn_qkv: the conversions happen inside the quantizer, the staging pass and the stores, so
the kernels' fp32 branches are compared with fp64 attention at the edges of tiles and for every store they have (two waves per
SIMD, the wide forward at head_dim 128 and 256, gradients of 32 and 64 rows per wave)."""
import math

import pytest
import torch

from helpers import assert_close
from oracle import oracle

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = [
    # B, H, Nq, Nk, D, causal
    (1, 4, 256, 256, 64, False),
    (1, 2, 1, 1, 64, False),
    (2, 3, 97, 131, 64, True),
    (1, 2, 65, 65, 128, True),
    (2, 2, 127, 300, 128, False),
    (1, 3, 33, 64, 256, True),
    (1, 2, 130, 70, 256, False),
    (2, 64, 520, 520, 128, True),      # 64 rows per wave in the backward
]


def _inputs(B, H, Nq, Nk, D, seed):
    g = torch.Generator().manual_seed(seed)
    mk = lambda n: torch.randn((B, H, n, D), generator=g) + 0.3 * torch.randn((B, H, n, 1), generator=g)
    return mk(Nq), mk(Nk), mk(Nk), torch.randn((B, H, Nq, D), generator=g)


def _check(qfa, q, k, v, do, causal, o, grads, heads):
    """heads: (batch, head) pairs that are compared"""
    sm = 1.0 / math.sqrt(q.shape[3])
    pick = lambda t: torch.stack([t[b, h] for b, h in heads])[None].cpu()
    qh, kh = (oracle.dequantize_per_token(*(pick(x) for x in qfa.quantize_for_attention(t)[:3]), torch.float64)
              for t in (q, k))
    v16, do16, o = pick(v).bfloat16(), pick(do).bfloat16(), pick(o)
    o_ref, _ = oracle.attn_fwd(qh, kh, v16, causal, sm)
    assert o.dtype == torch.float32
    # P enters the product in bf16 (2^-9 each); O itself is not rounded
    assert_close("O", o, o_ref, scaled=True, rel=2.0 ** -7)
    refs, spreads = oracle.attn_bwd(qh, kh, v16, do16, causal, sm, o=o.bfloat16(), spread=True)
    one_key = k.shape[2] == 1   # dQ and dK are zero there
    for name, got, want, sp in zip(("dQ", "dK", "dV"), grads, refs, spreads):
        assert got.dtype == torch.float32
        assert_close(name, pick(got), want, scaled=True, rel=2.0 ** -7, spread=sp,
                     cos_tol=-1.0 if one_key and name != "dV" else 0.999)


@pytest.mark.parametrize("B,H,Nq,Nk,D,causal", CASES)
def test_fp32_vs_oracle(qfa, B, H, Nq, Nk, D, causal):
    sm = 1.0 / math.sqrt(D)
    q, k, v, do = (t.to(DEV) for t in _inputs(B, H, Nq, Nk, D, seed=Nq + Nk + D))
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    o = qfa.quant_flash_attn_qkv(*leaves, causal, sm)
    grads = torch.autograd.grad(o, leaves, do)
    with torch.no_grad():
        assert torch.equal(o, qfa.quant_flash_attn_qkv(*leaves, causal, sm))
    q, k, v = (t.detach() for t in leaves)
    _check(qfa, q, k, v, do, causal, o.detach(), grads, [(0, 0), (B - 1, H - 1)])


def test_fp32_wide_forward_at_head_dim_128(qfa):
    """16 heads of 4096 x 4096 fill one round of the wide kernel's workgroups."""
    B, H, N, D, sm = 1, 16, 4096, 128, 128 ** -0.5
    q, k, v, do = (t.to(DEV) for t in _inputs(B, H, N, N, D, seed=5))
    o = qfa.quant_flash_attn_qkv(q, k, v, False, sm)
    qh, kh = (oracle.dequantize_per_token(*(x[:, 3:4].cpu() for x in qfa.quantize_for_attention(t)[:3]), torch.float64) for t in (q, k))
    o_ref, _ = oracle.attn_fwd(qh[:, :, 4000:].contiguous(), kh, v[:, 3:4].bfloat16().cpu(), False, sm)
    assert_close("O", o[:, 3:4, 4000:].cpu(), o_ref, scaled=True, rel=2.0 ** -7)


def test_fp32_strided_views_and_expanded_gradient(qfa):
    """[B,N,H,D] storage as permuted views, and a gradient that is one row expanded: the same bits as contiguous tensors."""
    B, H, N, D, sm = 2, 3, 100, 128, 0.09
    q, k, v, _ = (t.to(DEV) for t in _inputs(B, H, N, N, D, seed=9))
    do = torch.randn((1, 1, 1, D), generator=torch.Generator().manual_seed(1)).to(DEV).expand(B, H, N, D)

    def run(q, k, v, do):
        leaves = [t.requires_grad_(True) for t in (q, k, v)]
        o = qfa.quant_flash_attn_qkv(*leaves, True, sm)
        return (o.detach(),) + torch.autograd.grad(o, leaves, do)
    want = run(*(t.clone() for t in (q, k, v)), do.contiguous())
    got = run(*(t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3) for t in (q, k, v)), do)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_fp32_output_may_be_changed_in_place(qfa):
    """The backward does not read the fp32 output, which a caller may overwrite before it."""
    q, k, v, do = (t.to(DEV) for t in _inputs(1, 2, 70, 70, 64, seed=2))
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    want = torch.autograd.grad(qfa.quant_flash_attn_qkv(*leaves, True, 0.125), leaves, do)
    o = qfa.quant_flash_attn_qkv(*leaves, True, 0.125)
    o.detach().mul_(3.0)
    got = torch.autograd.grad(o, leaves, do)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
