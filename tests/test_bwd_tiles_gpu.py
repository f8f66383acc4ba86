"""The backward kernels at the edges of their tiles: one row less, as many and one more than a step of 32 and a tile of 64
streamed rows, the 64 (32) rows of a wave and the 256 (128) of a workgroup, with the first visible tile of a wave in any
place.  Against the closed-form gradients of the CPU oracle; the bar is the backward's (see helpers.py)."""
import math

import pytest
import torch

from test_attn_bwd_gpu import _check_grads, _fwd_bwd, _oracle_bwd
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
@pytest.mark.parametrize("H,Nq,Nk", [(2, 128, 128), (256, 256, 256), (256, 193, 300)])
@pytest.mark.parametrize("row", [0, 37, 70, 127])
def test_infinite_output_gradient_stays_with_the_keys_that_its_query_sees(qfa, D, dtype, H, Nq, Nk, row):
    """One dO row is infinite: dQ of the other queries stays finite, and so does dK of every key that the query does not see;
    dV of the key blocks of 32 that its block of 32 queries does not see at all (a block that the diagonal cuts multiplies
    the masked probabilities with it).  256 heads: 64 keys per wave at head_dim 128."""
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
