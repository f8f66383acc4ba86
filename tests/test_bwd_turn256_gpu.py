"""The backward at head_dim 256, whose tiles of 32 rows are waited for one turn after another: numbers of tiles around the three
buffers, ragged ends, and workgroups that run beside many others."""
import math

import pytest
import torch

from helpers import assert_close
from oracle import oracle

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Nq,Nk,causal", [(1, 1, True), (33, 32, False), (32, 33, False), (64, 64, True), (65, 96, True), (96, 65, False),
                                          (97, 129, False), (129, 129, True), (160, 161, False), (200, 517, True), (517, 200, False)])
def test_tiles_around_the_buffers(qfa, Nq, Nk, causal, dtype):
    """320 heads of the same values, more than the CUs take at once: the first against the oracle, the others bit for bit the same."""
    H, D, sm = 320, 256, 1.0 / 16.0
    g = torch.Generator().manual_seed(Nq * 1000 + Nk)
    mk = lambda n: (torch.randn((1, 1, n, D), generator=g) + 0.3 * torch.randn((1, 1, n, 1), generator=g)).to(dtype)
    q, k, v, do = mk(Nq), mk(Nk), mk(Nk), mk(Nq)
    leaves = [t.to(DEV).repeat(1, H, 1, 1).requires_grad_(True) for t in (q, k, v)]
    o = qfa.quant_flash_attn_qkv(*leaves, causal, sm)
    grads = torch.autograd.grad(o, leaves, do.to(DEV).repeat(1, H, 1, 1))
    qq, kq = (qfa.quantize_for_attention(t.to(DEV)) for t in (q, k))
    qh, kh = (oracle.dequantize_per_token(*(x.cpu() for x in t[:3]), torch.float64) for t in (qq, kq))
    refs, spreads = oracle.attn_bwd(qh, kh, v, do, causal, sm, o=o[:, :1].detach().cpu(), spread=True)
    for name, got, want, sp in zip(("dQ", "dK", "dV"), grads, refs, spreads):
        assert torch.equal(got, got[:, :1].expand_as(got)), f"{name}: heads of the same values differ"
        assert_close(name, got[:, :1].double().cpu(), want, scaled=True, rel=2.0 ** -7, spread=sp)
