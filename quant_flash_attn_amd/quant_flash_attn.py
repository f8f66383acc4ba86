"""INT8 per-token quantized flash attention -- drop-in for the reference's quant_flash_attn.py.

Two autograd entry points, both differentiable (the autograd nodes are native, csrc/qfa_torch.cpp) and backed by the HIP kernels behind qfa_attn_fwd / qfa_attn_bwd:

  QuantFlashAttnQKV.apply(q, k, v, causal, sm_scale)            (alias quant_flash_attn_qkv)
      Signature of the repository's fused-attention Function (flash_attn_triton.py:441).  Q and K
      are quantized per token inside (asymmetric_quant.py math), QK^T runs on INT8 MFMA, V stays
      in 16-bit.  Gradients flow straight through the quantizer to q and k.

  QuantFlashAttention.apply(q, kv_fp16, kv_quant, sm_scale)     (alias quant_flash_attn)
      The reference's own entry point (quant_flash_attn.py:173-240): one quantized tensor serves as
      K and V, `kv_fp16` only receives the gradient, backward returns (dq, dkv, None, None) with
      dkv = dK + dV (:161).  Query blocks of up to SHARED_KV_MAX_Q (512; 1024 at head_dim 256) tokens run the reference's
      computation itself in the forward (Q in 16-bit, qfa_attn_fwd_shared_kv) and in the backward
      (qfa_attn_bwd_shared_kv, binary16 arithmetic; bf16 tensors are converted around it).  Longer
      query blocks go through the INT8-score kernels, where Q is quantized per token too (stated
      difference from the reference, which keeps Q in fp16).
"""
from __future__ import annotations

from typing import Optional, Tuple

import torch

from . import _lib
from .asymmetric_quant import QuantizedTokens


def attn_fwd_quantized(qq: QuantizedTokens, kq: QuantizedTokens, v: torch.Tensor, causal: bool,
                       sm_scale: float, _entry: str = "qfa_attn_fwd") -> Tuple[torch.Tensor, torch.Tensor]:
    """O, LSE = attention(dequant(qq), dequant(kq), v).  v and O are bf16 or fp16 [B,H,N,D];
    LSE is fp32 [B,H,Nq] (natural log, as quant_flash_attn.py:79)."""
    # "qfa_bench_qk_stage" is the QK^T-only timing variant
    return _lib.host().attn_fwd(qq, kq, v, bool(causal), float(sm_scale), _entry == "qfa_bench_qk_stage")


def attn_bwd_quantized(qq: QuantizedTokens, kq: QuantizedTokens, v: torch.Tensor, o: torch.Tensor,
                       do: torch.Tensor, lse: torch.Tensor, causal: bool, sm_scale: float
                       ) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """dQ, dK, dV (w.r.t. the dequantized q^, k^ and v) in v's dtype."""
    return tuple(_lib.host().attn_bwd(qq, kq, v, o, do, lse, bool(causal), float(sm_scale)))


# Longest query block the shared-KV kernels are used for: they keep Q in 16 bits, and beat the INT8-score kernels while Nq is
# small against Nk -- the reference's test and benchmark shapes; crossover at Nk=4096, D=128 when the line was drawn: between
# 512 and 1024 queries (fwd 1.16 vs 1.51 ms at 512, 1.14 vs 1.01 ms at 1024; the tiled kernels have made the shared-KV side
# 1.8 times faster since, and the line stays because the two sides round differently).
SHARED_KV_MAX_Q = 512
# head_dim 256 (compute_flops.py:94): the INT8-score kernels run one wave per SIMD there and the crossover moves up
# (Nk=4096: fwd+bwd 5.9 vs 4.5 ms at 512 queries, 9.0 vs 8.9 at 1024; Nq=Nk=2048: 3.9 vs 4.9 ms, INT8-score first).
SHARED_KV_MAX_Q_BY_HEAD_DIM = {256: 1024}   # head_dim -> limit, where it differs from SHARED_KV_MAX_Q


def shared_kv_max_q(head_dim: int) -> int:
    """Longest query block that `quant_flash_attn` gives to the shared-KV kernels at this head_dim."""
    return SHARED_KV_MAX_Q_BY_HEAD_DIM.get(head_dim, SHARED_KV_MAX_Q)


def attn_fwd_shared_kv(q: torch.Tensor, codes: torch.Tensor, scale: torch.Tensor, zero_point: torch.Tensor,
                       sm_scale: float) -> Tuple[torch.Tensor, torch.Tensor]:
    """O, LSE = attention(q, kv, kv) with kv = (codes - zero_point) * scale, q in fp16 / bf16 and NOT
    quantized -- the computation of _attn_fwd_kernel_quantized (quant_flash_attn.py:22-83).
    O has q's dtype; LSE is fp32 [B,H,Nq] (natural log, :79)."""
    return _lib.host().skv_fwd(q, codes, scale, zero_point, float(sm_scale))


def attn_bwd_shared_kv(q: torch.Tensor, codes: torch.Tensor, scale: torch.Tensor, zero_point: torch.Tensor,
                       o: torch.Tensor, do: torch.Tensor, lse: torch.Tensor, sm_scale: float,
                       grad_dtype: Optional[torch.dtype] = None, grad_scale: Optional[torch.Tensor] = None
                       ) -> Tuple[torch.Tensor, torch.Tensor]:
    """dQ, dKV of attn_fwd_shared_kv: the computation of _attn_bwd_kernel_quantized
    (quant_flash_attn.py:104-166) with dKV = dV + dK as stored there (:161).  q, o, do fp16
    [B,H,Nq,D] (the kernels compute in binary16); lse as returned by the forward.  dQ and dKV come back
    in `grad_dtype` (fp16 by default, or bf16), multiplied by the one-element device tensor `grad_scale`
    if given.  Up to 32 queries (16 at head_dim 256), and 33 to 128 of many heads of 64 or 128, run in one
    fused pass over the codes, longer blocks in a dQ kernel plus a dKV kernel.  The keys are not split over
    workgroups here (`quant_flash_attn`'s backward does where there are few heads)."""
    return _lib.host().skv_bwd(q, codes, scale, zero_point, o, do, lse, float(sm_scale), grad_dtype or torch.float16,
                               grad_scale)


class QuantFlashAttnQKV:
    """apply(q, k, v, causal, sm_scale) -> o   (argument order of flash_attn_triton.py:441); backward -> (dq, dk, dv).

    q, k, v: [B,H,N,D] bf16 / fp16 / fp32 (fp32: V, dO and the O that the backward takes are rounded to bf16; where all three are
    fp32, O and the gradients are not).
    causal keeps key j for query i when j <= i (flash_attn_triton.py:50); with fewer queries than keys the mask is
    aligned to the last key (j <= i + Nk - Nq).
    With few (batch, head) pairs a head's keys (backward: streamed rows) are split over workgroups and their parts added in
    fp32: the last bits of a head's results depend on B * H, not on the other heads' values, and repeat from call to call."""

    @staticmethod
    def apply(q, k, v, causal, sm_scale):
        return _lib.host().qkv(q, k, v, bool(causal), float(sm_scale))


quant_flash_attn_qkv = QuantFlashAttnQKV.apply


class QuantFlashAttnQuantizedKV:
    """apply(q, k_fp16, v_fp16, k_quant, v_quant, causal, sm_scale) -> o; backward -> (dq, dk, dv).

    The reference's contract (quant_flash_attn.py:178-237: the keys and values arrive as INT8 codes with per-token
    scale and zero point, a 16-bit placeholder leaf receives the gradient) with K and V as two separately quantized
    tensors instead of one shared tensor, and a causal flag.  k_quant and v_quant are (codes, scale, zero_point)
    tuples as asymmetric_quant_per_token returns them; k_fp16 and v_fp16 are only placeholders.
    Short query blocks (decoding) run in one pass over the cache (qfa_attn_fwd_cache), with V as its exact codes.  In longer
    ones the K codes are used as they are (INT8 scores) and V is dequantized once per call by the HIP dequantizer into a
    16-bit tensor that the P.V product streams: converting int8 V inside that kernel would add about 56 vector
    instructions per 32x32 block to a loop that issues 83 and is bound by them, the separate pass adds
    a read of the codes and one 16-bit write and read (8 % of the forward at B4 H32 N4096 D128).  With and without a
    gradient the result is the same, bit for bit; the keys are split as in QuantFlashAttnQKV."""

    @staticmethod
    def apply(q, k_fp16, v_fp16, k_quant, v_quant, causal, sm_scale):
        kc, ks, kz = k_quant
        vc, vs, vz = v_quant
        return _lib.host().cache(q, k_fp16, v_fp16, kc, ks, kz, vc, vs, vz, bool(causal), float(sm_scale))


quant_flash_attn_quantized_kv = QuantFlashAttnQuantizedKV.apply


class QuantFlashAttention:
    """apply(q, kv_fp16, kv_quant, sm_scale) -> o; backward -> (dq, dkv).

    Positional contract of the reference (quant_flash_attn.py:178-237): kv_quant is the
    (codes, scale, zero_point) tuple returned by asymmetric_quant_per_token, kv_fp16 is only a
    placeholder leaf that receives dkv, attention is non-causal, K == V == dequant(kv_quant).  The keys are split as in
    QuantFlashAttnQKV."""

    @staticmethod
    def apply(q, kv_fp16, kv_quant, sm_scale):
        codes, scale, zp = kv_quant
        return _lib.host().shared(q, kv_fp16, codes, scale, zp, float(sm_scale), shared_kv_max_q(q.shape[-1]))


def _normalised_dout(grad_output: torch.Tensor, kv_scale: torch.Tensor):
    """(dO * 2^k as float16, 2^-k as a one-element float32 tensor) for the binary16 backward kernels
    (qfa_dout_normalise: two launches, nothing synchronises).

    k puts the largest |dO| * 2^k * (largest key scale) into (4, 8]: 2^8 for |dO| when the key scales are of the usual
    size (2^-5 for values of order one), higher when they are smaller and lower when they are larger, since the operands
    the kernels form carry the key scale as a factor (ds * scale_j must neither sink into binary16's subnormals nor
    leave its range); dO * 2^k itself stays at or below 2^14."""
    return _lib.host().normalised_dout(grad_output, kv_scale)


quant_flash_attn = QuantFlashAttention.apply
