"""The forward kernel with one wave per SIMD (head_dim 256, and long unmasked sequences at 128) at the edges of its tiles:
around a step of 32 and a tile of 64 keys, the 32 (64) queries of a wave and the 128 (256) of a workgroup.  Against fp64
attention on the dequantized inputs; the bar is the forward's (see helpers.py)."""
import math

import pytest
import torch

from helpers import assert_close, max_abs
from quant_flash_attn_amd.synthetic import make_inputs
from test_attn_fwd_gpu import LSE_TOL, _oracle_fwd, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Nq,Nk,causal", [(1, 1, False), (31, 33, True), (32, 64, False), (33, 127, True), (63, 129, False),
                                          (64, 255, True), (65, 257, False), (96, 256, True), (129, 129, True), (161, 513, True)])
def test_head_dim_256_at_tile_edges(qfa, Nq, Nk, causal, dtype):
    q, k, v, _ = make_inputs("offset", 1, 3, Nk, 256, seed=Nq + 7 * Nk, dtype=dtype)
    q = q[:, :, :Nq].contiguous()
    qq, kq, o, lse = _run(qfa, q, k, v, causal, 1.0 / 16)
    o_ref, lse_ref = _oracle_fwd(qq, kq, v, causal, 1.0 / 16)
    assert_close("O", o.cpu(), o_ref)
    assert max_abs(lse.cpu(), lse_ref) < LSE_TOL


# sizes that fill a round of 256 workgroups of 256 queries: whole ones, a ragged last tile of keys, and 245 of 256 rows
# (bnhd: codes and V stored token by token and handed over as permuted views)
@pytest.mark.parametrize("H,Nq,Nk,jump", [(256, 256, 4096, 0), (128, 512, 4127, 0), (256, 245, 4161, 0), (256, 256, 4096, 300)])
@pytest.mark.parametrize("dtype,layout", [(torch.bfloat16, "bhnd"), (torch.float16, "bhnd"), (torch.bfloat16, "bnhd")])
def test_long_unmasked_head_dim_128(qfa, H, Nq, Nk, jump, dtype, layout):
    q, k, v, _ = make_inputs("offset", 1, H, Nk, 128, seed=Nq + Nk, dtype=dtype)
    q = q[:, :, :Nq].contiguous()
    if jump:   # keys whose scores exceed all before them by more than the running sums can hold
        k[:, :, 2000:2010] *= jump
    sm = 1.0 / math.sqrt(128)
    if layout == "bhnd":
        qq, kq, o, lse = _run(qfa, q, k, v, False, sm)
    else:
        turn = lambda t: t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)   # noqa: E731
        qq, kq = (x._replace(codes=turn(x.codes)) for x in (qfa.quantize_for_attention(t.to("cuda:0")) for t in (q, k)))
        o, lse = qfa.attn_fwd_quantized(qq, kq, turn(v.to("cuda:0")), False, sm)
    for h in (0, H // 2 + 1, H - 1):
        o_ref, lse_ref = _oracle_fwd(qq, kq, v, False, sm, heads=(0, h))
        assert_close("O", o[:, h:h + 1].cpu(), o_ref)
        # (relative where the scores are large: fp32 products of scores of that size)
        assert max_abs(lse[:, h:h + 1].cpu(), lse_ref) < LSE_TOL + 2.0 ** -21 * float(lse_ref.abs().max())
