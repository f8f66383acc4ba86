"""The backward kernels at the edges of their tiles: one row less, as many and one more than a step of 32 and a tile of 64
streamed rows, the 32 rows of a wave and the 128 of a workgroup (few heads) and, at head_dim 128 with many heads, the 64 of a
wave and the 256 of a workgroup, with the first visible tile of a wave in any place.  Against the closed-form gradients of
the CPU oracle; the bar is the backward's (see helpers.py)."""
import math

import pytest
import torch

from test_attn_bwd_gpu import DEV, _check_grads, _fwd_bwd, _oracle_bwd
from quant_flash_attn_amd.synthetic import make_inputs


@pytest.mark.gpu
@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.bfloat16), (256, torch.bfloat16)])
@pytest.mark.parametrize("Nq,Nk,causal", [(1, 1, False), (31, 33, True), (32, 64, False), (33, 127, True), (63, 129, False),
                                          (64, 255, True), (65, 257, False), (96, 256, True), (257, 257, True), (161, 513, True)])
def test_backward_at_tile_edges(qfa, Nq, Nk, causal, D, dtype):
    q, k, v, do = make_inputs("offset", 1, 3, max(Nq, Nk), D, seed=Nq + 7 * Nk + D, dtype=dtype)
    q, do = q[:, :, :Nq].contiguous(), do[:, :, :Nq].contiguous()
    k, v = k[:, :, :Nk].contiguous(), v[:, :, :Nk].contiguous()
    sm = 1.0 / math.sqrt(D)
    qq, kq, o, _, dq, dk, dv = _fwd_bwd(qfa, q, k, v, do, causal, sm)
    want, spreads = _oracle_bwd(qq, kq, v, do, o, causal, sm)
    _check_grads("", (dq.cpu(), dk.cpu(), dv.cpu()), want, spreads)


# 256 heads at head_dim 128: the sizes at which both kernels, or the one named, take 64 rows per wave
@pytest.mark.gpu
@pytest.mark.parametrize("dtype,layout", [(torch.bfloat16, "bhnd"), (torch.float16, "bhnd"), (torch.bfloat16, "bnhd")])
@pytest.mark.parametrize("Nq,Nk,causal", [(63, 129, False),     # dK / dV
                                          (128, 256, True),     # dK / dV
                                          (161, 513, True), (511, 515, True),   # dQ
                                          (193, 300, False), (257, 257, False), (512, 512, False), (200, 200, True),
                                          (256, 256, True), (449, 449, True),
                                          (512, 512, True), (420, 512, True)])
def test_64_rows_per_wave(qfa, Nq, Nk, causal, dtype, layout):
    B, H, D = 2, 128, 128
    q, k, v, do = make_inputs("offset", B, H, Nk, D, seed=Nq + 3 * Nk, dtype=dtype)
    q, do = q[:, :, :Nq].contiguous(), do[:, :, :Nq].contiguous()
    sm = 1.0 / math.sqrt(D)
    # token-major storage handed over as permuted views: codes, V, O and dO
    turn = (lambda t: t) if layout == "bhnd" else (lambda t: t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3))
    qq, kq = (x._replace(codes=turn(x.codes)) for x in (qfa.quantize_for_attention(t.to(DEV)) for t in (q, k)))
    vg, dog = turn(v.to(DEV)), turn(do.to(DEV))
    o, lse = qfa.attn_fwd_quantized(qq, kq, vg, causal, sm)
    o = turn(o)
    grads = qfa.attn_bwd_quantized(qq, kq, vg, o, dog, lse, causal, sm)
    for b, h in ((0, 0), (0, 101), (1, 127)):
        want, spreads = _oracle_bwd(qq, kq, v, do, o, causal, sm, b, h)
        _check_grads(f" head {b},{h}", [g[b:b + 1, h:h + 1].cpu() for g in grads], want, spreads)


@pytest.mark.gpu
@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.bfloat16), (256, torch.bfloat16)])
def test_infinite_value_row_stays_with_the_queries_that_see_it(qfa, D, dtype):
    """The last key's V row is infinite: O and dQ of the query blocks of 32 that end before it stay finite (a block that
    the diagonal cuts multiplies the masked probabilities with it)."""
    N = 128
    q, k, v, do = make_inputs("normal", 1, 2, N, D, seed=D, dtype=dtype)
    v[:, :, -1] = float("inf")
    _, _, o, _, dq, _, _ = _fwd_bwd(qfa, q, k, v, do, True, 1.0 / math.sqrt(D))
    assert torch.isfinite(o[:, :, :96].float()).all() and torch.isfinite(dq[:, :, :96].float()).all()
    assert not torch.isfinite(o[:, :, -1].float()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.bfloat16), (256, torch.bfloat16)])
@pytest.mark.parametrize("H,Nq,Nk", [(2, 128, 128), (256, 128, 256), (256, 449, 449), (256, 193, 300)])
@pytest.mark.parametrize("row", [0, 37, 70, 127])
def test_infinite_output_gradient_stays_with_the_keys_that_its_query_sees(qfa, D, dtype, H, Nq, Nk, row):
    """One dO row is infinite: dQ of the other queries stays finite, and so does dK of every key that the query does not see;
    dV of the key blocks of 32 that its block of 32 queries does not see at all (a block that the diagonal cuts multiplies
    the masked probabilities with it).  256 heads of 128: 64 keys per wave at the first two of their sizes."""
    q, k, v, do = make_inputs("normal", 1, H, Nk, D, seed=D + row, dtype=dtype)
    q, do = q[:, :, :Nq].contiguous(), do[:, :, :Nq].contiguous()
    do[:, :, row] = float("inf")
    _, _, _, _, dq, dk, dv = _fwd_bwd(qfa, q, k, v, do, True, 1.0 / math.sqrt(D))
    off = Nk - Nq
    block = (row // 32 * 32 + 31 + off) // 32 * 32 + 32   # first key block behind what the query's block sees
    others = [i for i in range(Nq) if i != row]
    assert torch.isfinite(dq[:, :, others].float()).all()
    assert torch.isfinite(dk[:, :, row + off + 1:].float()).all()
    assert torch.isfinite(dv[:, :, block:].float()).all()
    assert not torch.isfinite(dv[:, :, :row + off + 1].float()).all()
