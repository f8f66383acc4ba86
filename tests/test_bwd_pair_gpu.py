"""dK / dV and dQ in one launch whose two kinds of workgroups are divided differently: other rows per wave, other numbers of parts, one
kind divided and the other not.  Against fp64 attention on the dequantized Q and K."""
import math

import pytest
import torch

from helpers import assert_close
from oracle import oracle
from plans import bwd_plan
from test_bwd_split_gpu import _inputs

CASES = [
    # B, H, Nq, Nk, D, causal, dtype, rows per wave / 32 and parts of dK / dV, of dQ
    (1, 1, 327, 327, 128, False, torch.bfloat16, (1, 6, 1, 3)),
    (1, 12, 279, 2790, 128, True, torch.bfloat16, (2, 1, 1, 3)),
    (2, 20, 1500, 200, 128, False, torch.float16, (1, 3, 2, 1)),
    (2, 20, 64, 1500, 128, True, torch.float16, (2, 1, 1, 6)),
    (1, 1, 197, 564, 64, True, torch.float32, (1, 4, 1, 3)),
    (1, 1, 304, 304, 64, False, torch.bfloat16, (1, 5, 1, 5)),
    (1, 1, 289, 289, 256, True, torch.bfloat16, (1, 5, 1, 1)),
    (1, 1, 303, 303, 256, False, torch.float16, (1, 5, 1, 2)),
]


@pytest.mark.parametrize("B,H,Nq,Nk,D,causal,dtype,plan", CASES)
def test_the_plan_divides_them_so(B, H, Nq, Nk, D, causal, dtype, plan):
    p = bwd_plan(B * H, Nq, Nk, D, causal)
    assert (p.blocks_dkv, p.splits_dkv, p.blocks_dq, p.splits_dq) == plan


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Nq,Nk,D,causal,dtype,plan", CASES)
def test_both_kinds_in_one_launch(qfa, B, H, Nq, Nk, D, causal, dtype, plan):
    sm = 1.0 / math.sqrt(D)
    q, k, v, do = _inputs(B, H, Nq, Nk, D, dtype)
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    o = qfa.quant_flash_attn_qkv(*leaves, causal, sm)
    grads = torch.autograd.grad(o, leaves, do)
    io = torch.bfloat16 if dtype == torch.float32 else dtype
    v16, o16, do16 = (t.detach().to(io).cpu() for t in (v, o, do))
    qh, kh = (oracle.dequantize_per_token(*(x.cpu() for x in qfa.quantize_for_attention(t.detach())[:3]), torch.float64) for t in (q, k))
    refs, spreads = oracle.attn_bwd(qh, kh, v16, do16, causal, sm, o=o16, spread=True)
    for name, got, want, sp in zip(("dQ", "dK", "dV"), grads, refs, spreads):
        assert_close(name, got.double().cpu(), want, scaled=True, rel=2.0 ** -7, spread=sp)   # (as the split backward's)
