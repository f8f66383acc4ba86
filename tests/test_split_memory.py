"""The memory of the INT8-score kernels' parts where their streamed rows are dealt to several workgroups: bounded, shared by dK / dV
and dQ where both are large, and not needed where it is not there."""
import gc
import math
import random

import pytest
import torch

from plans import bwd_plan
from quant_flash_attn_amd import _lib
from test_bwd_split_gpu import _inputs, _parts, _undivided

DEV = "cuda:0"
MIB = 1 << 20


def _same(grads, whole):
    """The same products of the same operands, added in another order and rounded once more or less (2^-8 in bf16); the two LSE
    differ by the rounding of the probabilities that they sum (2^-9)."""
    for name, got, un in zip(("dQ", "dK", "dV"), grads, whole):
        assert torch.isfinite(got).all(), name
        diff = (got.double() - un.double()).norm() / un.double().norm()
        assert diff < 2.0 ** -7, f"{name}: {float(diff)}"


def test_parts_are_bounded():
    """At most QFA_SPLIT_PART_BYTES (224 MiB) of parts in the forward, and in the backward, whatever the sizes."""
    L, rng, most = _lib.lib(), random.Random(3), [0, 0]
    log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    shapes = [(1, 2, 16384, 16384, 256, 1), (1, 200, 256, 30000, 256, 0), (1, 2, 22030, 22030, 256, 1)]
    for _ in range(20000):
        Nk = log(1, 40000)
        shapes.append((log(1, 16), log(1, 128), Nk if rng.random() < 0.6 else log(1, Nk), Nk, rng.choice((64, 128, 256)), rng.randint(0, 1)))
    for s in shapes:
        fwd, bwd = L.qfa_attn_fwd_split_workspace_bytes(*s), _parts(*s)
        assert 0 <= fwd <= 224 * MIB and 0 <= bwd <= 224 * MIB, s
        most = [max(most[0], fwd), max(most[1], bwd)]
    assert min(most) > 96 * MIB   # (the sample comes near the bound)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Nq,Nk,D,causal,dtype", [(1, 2, 8319, 8319, 256, True, torch.bfloat16), (1, 2, 8448, 8448, 256, False, torch.float32),
                                                      (2, 3, 6803, 6803, 128, True, torch.float16)])
def test_parts_of_dq_in_the_place_of_the_others(qfa, B, H, Nq, Nk, D, causal, dtype):
    """Parts of both beyond 128 MiB together: the gradients of the undivided call, and again on buffers that hold what the first
    pass left."""
    plan = bwd_plan(B * H, Nq, Nk, D, causal)
    assert plan.sum_between and plan.splits_dkv > 1 and plan.splits_dq > 1 and plan.part_bytes == _parts(B, H, Nq, Nk, D, causal)
    sm = 1.0 / math.sqrt(D)
    q, k, v, do = _inputs(B, H, Nq, Nk, D, dtype)
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    grads = None
    for _ in range(2):
        o = qfa.quant_flash_attn_qkv(*leaves, causal, sm)
        again = torch.autograd.grad(o, leaves, do)
        assert grads is None or all(torch.equal(a, b) for a, b in zip(grads, again))
        grads = again
    q, k, v, o = (t.detach() for t in (q, k, v, o))
    io = torch.bfloat16 if dtype == torch.float32 else dtype
    v16, o16, do16 = (t.to(io) for t in (v, o, do))
    qq, kq = qfa.quantize_for_attention(q), qfa.quantize_for_attention(k)
    whole = _undivided(qq, kq, v16, o16, do16, qfa.attn_fwd_quantized(qq, kq, v16, causal, sm)[1], causal, sm)
    _same(grads, whole)


def _limited(f, parts):
    """f() with all memory, and with half of `parts` bytes less than it took beyond what was held at its start.  Both times holes in
    the held memory that the parts could lie in are filled first: what earlier tests left there decides neither."""
    res, total = [], torch.cuda.get_device_properties(0).total_memory
    for limited in (False, True):
        gc.collect()
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        held, plugs = torch.cuda.memory_reserved(), []
        try:
            torch.cuda.set_per_process_memory_fraction(held / total)
            try:
                while True:
                    plugs.append(torch.empty(parts // 2, dtype=torch.uint8, device=DEV))
            except torch.OutOfMemoryError:
                pass
            torch.cuda.set_per_process_memory_fraction((held + taken - parts // 2) / total if limited else 1.0)
            torch.cuda.reset_peak_memory_stats()
            res.append([t.cpu() for t in f()])
            taken = torch.cuda.max_memory_reserved() - held
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
    return res


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_without_memory_for_the_parts(qfa, dtype):
    """Half of the parts' memory is missing: forward and backward run undivided."""
    gc.collect()
    torch.cuda.empty_cache()
    B, H, N, D, sm, io = 1, 2, 8000, 256, 1.0 / 16, torch.bfloat16
    q, k, v, do = _inputs(B, H, N, N, D, dtype)
    fwd, bwd = _lib.lib().qfa_attn_fwd_split_workspace_bytes(B, H, N, N, D, 1), _parts(B, H, N, N, D, True)
    assert min(fwd, bwd) > 32 * MIB
    with torch.no_grad():
        o, o_limited = (r[0] for r in _limited(lambda: [qfa.quant_flash_attn_qkv(q, k, v, True, sm)], fwd))
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    out = qfa.quant_flash_attn_qkv(*leaves, True, sm)
    grads, grads_limited = _limited(lambda: torch.autograd.grad(out, leaves, do, retain_graph=True), bwd)
    qq, kq = qfa.quantize_for_attention(q.detach()), qfa.quantize_for_attention(k.detach())
    whole = qfa.attn_fwd_quantized(qq, kq, v.detach().to(io), True, sm)[0].cpu()
    assert torch.equal(o_limited.to(io), whole) and not torch.equal(o.to(io), whole)
    assert not any(torch.equal(a, b) for a, b in zip(grads, grads_limited))
    _same(grads_limited, grads)
