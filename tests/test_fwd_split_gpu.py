"""The INT8-score forward with its keys split over workgroups (few queries, many keys), against fp64 attention on the dequantized
Q and K and against the kernel that does not split: parts without a visible key, ragged ends, rows whose maximum comes late."""
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
    (1, 2, 1, 1000, 64, True, torch.bfloat16),
    (1, 3, 129, 4033, 64, True, torch.float16),       # a block of one query, one key in the last tile
    (2, 2, 1500, 1500, 64, True, torch.bfloat16),     # the first queries see nothing of the later parts
    (1, 4, 333, 7001, 128, True, torch.bfloat16),     # parts that only some rows of a wave see
    (1, 2, 200, 3000, 128, False, torch.float16),
    (2, 1, 1000, 1000, 128, True, torch.float32),
    (1, 2, 1100, 1100, 256, True, torch.bfloat16),
    (1, 3, 97, 2049, 256, True, torch.float16),
    (1, 1, 260, 1501, 256, False, torch.float32),
]


def _workspace(B, H, Nq, Nk, D, causal):
    return _lib.lib().qfa_attn_fwd_split_workspace_bytes(B, H, Nq, Nk, D, int(causal))


def _rows(Nq):   # a sample with the edges of waves and blocks
    return sorted({r for r in (0, 1, 31, 32, 63, 64, 127, 128, 255, 256, Nq // 2, Nq - 2, Nq - 1) if 0 <= r < Nq})


@pytest.mark.parametrize("late", [False, True])
@pytest.mark.parametrize("B,H,Nq,Nk,D,causal,dtype", CASES)
def test_split_forward(qfa, B, H, Nq, Nk, D, causal, dtype, late):
    assert _workspace(B, H, Nq, Nk, D, causal) > 0, "the plan splits this shape"
    sm = 1.0 / math.sqrt(D)
    g = torch.Generator().manual_seed(Nq + Nk + D)
    mk = lambda n: torch.randn((B, H, n, D), generator=g) + 0.3 * torch.randn((B, H, n, 1), generator=g)
    q, k, v = mk(Nq), mk(Nk), mk(Nk)
    if late:   # scores a hundred times as large from the middle on: references move while other rows see no key
        k[:, :, Nk // 2:] *= 100.0
    q, k, v = (t.to(dtype).to(DEV) for t in (q, k, v))
    v16 = v.bfloat16() if dtype == torch.float32 else v
    with torch.no_grad():
        o = qfa.quant_flash_attn_qkv(q, k, v, causal, sm)
        qq, kq = qfa.quantize_for_attention(q), qfa.quantize_for_attention(k)
        whole, _ = qfa.attn_fwd_quantized(qq, kq, v16, causal, sm)
    assert o.dtype == dtype and torch.isfinite(o).all()
    # the same probabilities but for their rounding to 16 bits, 2^-9 of each in bf16; O the same once more
    assert_close("O against the whole", o.double().cpu(), whole.double().cpu(), scaled=True, rel=2.0 ** -7)
    r = _rows(Nq)
    qh, kh = (oracle.dequantize_per_token(*(x[-1:, -1:].cpu() for x in t[:3]), torch.float64) for t in (qq, kq))
    for i in r:
        n = Nk - Nq + i + 1 if causal else Nk
        o_ref, _ = oracle.attn_fwd(qh[:, :, i:i + 1], kh[:, :, :n], v16[-1:, -1:, :n].cpu(), False, sm)
        assert_close(f"O, row {i}", o[-1:, -1:, i:i + 1].double().cpu(), o_ref, scaled=True, rel=2.0 ** -7)


def test_split_forward_keeps_what_a_backward_takes(qfa):
    """O of a call that keeps its tensors for a backward is the same bits, and the gradients are those of its LSE."""
    B, H, Nq, Nk, D, sm = 1, 2, 700, 1500, 128, 0.09
    assert _workspace(B, H, Nq, Nk, D, True) > 0
    for dtype in (torch.bfloat16, torch.float32):
        g = torch.Generator().manual_seed(3)
        # [B,N,H,D] storage
        q, k, v, do = (torch.randn((B, n, H, D), generator=g).to(dtype).to(DEV).transpose(1, 2) for n in (Nq, Nk, Nk, Nq))
        with torch.no_grad():
            o = qfa.quant_flash_attn_qkv(q, k, v, True, sm)
        leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
        o2 = qfa.quant_flash_attn_qkv(*leaves, True, sm)
        assert torch.equal(o, o2)
        grads = torch.autograd.grad(o2, leaves, do)
        qh, kh = (oracle.dequantize_per_token(*(x.cpu() for x in qfa.quantize_for_attention(t)[:3]), torch.float64) for t in (q, k))
        v16, do16, o16 = (t.bfloat16().cpu() for t in (v, do, o))
        refs, spreads = oracle.attn_bwd(qh, kh, v16, do16, True, sm, o=o16, spread=True)
        for name, got, want, sp in zip(("dQ", "dK", "dV"), grads, refs, spreads):
            assert_close(name, got.cpu(), want, scaled=True, rel=2.0 ** -7, spread=sp)


def test_split_forward_replayed_from_a_graph(qfa):
    """The partial results are workspace of the call: every replay of a captured call gives the eager bits."""
    g = torch.Generator().manual_seed(4)
    q, k, v = (torch.randn((1, 4, n, 128), generator=g).bfloat16().to(DEV) for n in (100, 4000, 4000))
    with torch.no_grad():
        want = qfa.quant_flash_attn_qkv(q, k, v, True, 0.09)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = qfa.quant_flash_attn_qkv(q, k, v, True, 0.09)
        for i in range(3):
            got.zero_()
            graph.replay()
            assert torch.equal(got, want)
            q.neg_()
            want = qfa.quant_flash_attn_qkv(q, k, v, True, 0.09)
            torch.cuda.synchronize()


@pytest.mark.parametrize("D", [64, 128, 256])
def test_nan_keys_stay_with_the_queries_that_see_them(qfa, D):
    """A part of the keys in which some queries of a wave see NaN keys only and the others none: those others keep their rows."""
    B, H, Nq, Nk, sm = 1, 2, 1090, 1100, 1.0 / math.sqrt(D)   # query i sees keys up to i + 10: parts begin inside a wave's triangle
    rows = B * H * Nq * (D + 2) * 4
    splits = _workspace(B, H, Nq, Nk, D, True) // rows
    assert splits > 1, "the plan splits this shape"
    part = -(-((Nk + 63) // 64) // splits) * 64
    g = torch.Generator().manual_seed(D)
    q, k, v = (torch.randn((B, H, n, D), generator=g).bfloat16().to(DEV) for n in (Nq, Nk, Nk))
    (kc, ks, kz), vq, none = qfa.asymmetric_quant_per_token(k), qfa.asymmetric_quant_per_token(v), torch.empty(0, device=DEV)
    with torch.no_grad():
        want = qfa.quant_flash_attn_quantized_kv(q, none, none, (kc, ks, kz), vq, True, sm)
        ks = ks.clone()
        ks[:, :, part:] = float("nan")
        got = qfa.quant_flash_attn_quantized_kv(q, none, none, (kc, ks, kz), vq, True, sm)
    first = part - (Nk - Nq)   # the first query that sees a NaN key
    assert torch.isnan(got[:, :, first:]).all()
    # (a wave's references may move at other tiles: the probabilities are rounded against another one)
    assert_close("O", got[:, :, :first].cpu(), want[:, :, :first].double().cpu(), scaled=True, rel=2.0 ** -7)
