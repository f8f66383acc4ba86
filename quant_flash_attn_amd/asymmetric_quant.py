"""Per-token asymmetric INT8 quantization -- drop-in for the reference's asymmetric_quant.py.

`asymmetric_quant_per_token(x)` keeps the reference's name, argument and return structure
(asymmetric_quant.py:109-149): codes int8 [B,H,N,D], scale [B,H,N,1] (fp16 by default, as the
reference stores it, :128), zero point int8 [B,H,N,1].  The work is done by the HIP kernel
behind qfa_quant_per_token; `quantize_for_attention` additionally returns the fp32 scale and
the per-token code sums that the INT8 attention kernels consume.
"""
from __future__ import annotations

from typing import NamedTuple, Tuple

import torch

from . import _lib


class QuantizedTokens(NamedTuple):
    codes: torch.Tensor      # int8  [B,H,N,D]
    scale: torch.Tensor      # fp32  [B,H,N,1]  (the scale the codes were computed with)
    zero_point: torch.Tensor  # int8  [B,H,N,1]
    rowsum: torch.Tensor     # int32 [B,H,N,1]  sum of the token's codes


def asymmetric_quant_per_token(input_tensor: torch.Tensor, scale_dtype: torch.dtype = torch.float16
                               ) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """Quantizes a (Batch, Heads, Seq, Head_Dim) tensor to INT8, one scale / zero point per token.

    Same contract as the reference's function of this name (asymmetric_quant.py:109-149).
    Returns (codes int8 [B,H,N,D], scale [B,H,N,1] of `scale_dtype`, zero_point int8 [B,H,N,1]).
    The codes are computed with the unrounded fp32 scale; the returned scale is its
    round-to-nearest cast (fp16 by default like the reference; pass torch.float32 to keep it).
    """
    return _lib.host().quant(input_tensor, scale_dtype)


def quantize_for_attention(x: torch.Tensor) -> QuantizedTokens:
    """Quantizes like asymmetric_quant_per_token and also returns what the INT8 attention kernels
    need beside the codes: the fp32 scale and the per-token sum of the codes."""
    return QuantizedTokens(*_lib.host().quant_attn(x))


def quantize_pair_for_attention(x0: torch.Tensor, x1: torch.Tensor) -> Tuple[QuantizedTokens, QuantizedTokens]:
    """quantize_for_attention of two tensors (the queries and the keys of an attention call: same batch, heads,
    head dimension and element type, any two lengths) in ONE launch; bit-identical to two separate calls."""
    a, b = _lib.host().quant_attn_pair(x0, x1)
    return QuantizedTokens(*a), QuantizedTokens(*b)


def dequantize_per_token(codes: torch.Tensor, scale: torch.Tensor, zero_point: torch.Tensor,
                         dtype: torch.dtype = torch.float32) -> torch.Tensor:
    """(codes - zero_point) * scale per token (the reference's dequantize_per_token_torch,
    asymmetric_quant.py:158-160), as a HIP kernel writing `dtype`."""
    return _lib.host().dequant(codes, scale, zero_point, dtype)


def code_rowsum(codes: torch.Tensor) -> torch.Tensor:
    """int32 [B,H,N,1] sum of each token's codes (what quantize_for_attention emits beside the codes), as a HIP
    kernel, for codes that arrive already quantized."""
    return _lib.host().rowsum(codes)
