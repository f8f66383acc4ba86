"""dK / dV and dQ in one launch whose two kinds of workgroups are divided differently: other rows per wave, other numbers of parts, one
kind divided and the other not.  Against fp64 attention on the dequantized Q and K."""
import math
import re

import pytest
import torch

from helpers import assert_close, launches
from oracle import oracle
from plans import bwd_plan, bwd_plan_within
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


def _workgroups(BH, rows, blocks, splits):
    return (BH * -(-rows // (128 * blocks)) + 7) // 8 * 8 * splits


LAUNCHED = [
    # heads, Nq, Nk, D, causal: undivided, with other rows per wave than either kind would take by itself; then divided; then a full chip
    (7, 1542, 4268, 128, False), (15, 782, 2179, 128, True), (6, 3420, 3420, 128, False), (170, 1056, 1056, 128, False),
    (12, 279, 2790, 128, True), (3, 1866, 1866, 64, True), (2, 1936, 1936, 256, False), (96, 691, 691, 128, True),
]


@pytest.mark.gpu
@pytest.mark.parametrize("H,Nq,Nk,D,causal", LAUNCHED)
def test_the_planned_division_is_launched(qfa, H, Nq, Nk, D, causal):
    p = bwd_plan(H, Nq, Nk, D, causal)
    *leaves, do = _inputs(1, H, Nq, Nk, D, torch.bfloat16)
    for t in leaves:
        t.requires_grad_(True)
    names = launches(lambda: qfa.quant_flash_attn_qkv(*leaves, causal, 0.1), lambda o: torch.autograd.grad(o, leaves, do, retain_graph=True))
    pair, = (x for x in names if "bwd_pair_kernel" in x[0])
    assert [int(x) for x in re.findall(r"Li(\d+)E", pair[0])] == [D, p.blocks_dkv, p.blocks_dq], pair
    assert pair[1] == _workgroups(H, Nk, p.blocks_dkv, p.splits_dkv) + _workgroups(H, Nq, p.blocks_dq, p.splits_dq), pair
    assert any("bwd_sum_kernel" in x[0] for x in names) == (p.part_bytes > 0)


@pytest.mark.gpu
@pytest.mark.parametrize("H,Nq,Nk,causal", [(170, 1056, 1056, False), (15, 782, 2179, True), (6, 3420, 3420, False)])
def test_rows_per_wave_do_not_change_the_bits(qfa, H, Nq, Nk, causal):
    """The undivided call and its heads one by one, whose rows per wave are others."""
    q, k, v, do = _inputs(1, H, Nq, Nk, 128, torch.bfloat16)
    qq, kq = qfa.quantize_for_attention(q), qfa.quantize_for_attention(k)
    o, lse = qfa.attn_fwd_quantized(qq, kq, v, causal, 0.1)
    whole = qfa.attn_bwd_quantized(qq, kq, v, o, do, lse, causal, 0.1)
    one, all_ = (bwd_plan_within(n, Nq, Nk, 128, causal, 0) for n in (1, H))
    assert (one.blocks_dkv, one.blocks_dq) != (all_.blocks_dkv, all_.blocks_dq)
    for h in (0, H // 2, H - 1):
        cut = lambda t: t[:, h:h + 1].contiguous()   # noqa: E731
        part = qfa.attn_bwd_quantized(type(qq)(*map(cut, qq)), type(kq)(*map(cut, kq)), cut(v), cut(o), cut(do), cut(lse), causal, 0.1)
        for name, got, want in zip(("dQ", "dK", "dV"), part, whole):
            assert torch.equal(got, cut(want)), (name, h)
