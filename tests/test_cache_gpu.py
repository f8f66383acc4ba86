"""qfa_attn_fwd_cache: short query blocks on an INT8 cache, through quant_flash_attn_quantized_kv, against the fp64 oracle
on exactly the quantized operands (the queries' codes from the C oracle of the quantizer).

Bound per element: the probabilities times the value scale are rounded to binary16 before the P.V product (2^-11 each, so
at most 2^-11 sum_j p_j |v_jd| in the output; a factor 2 covers the fp32 exponentials), the output is rounded once, and
the codes enter the fp32 sums with an offset (at most 1152 + 255 per key) that is subtracted at the end: 32 roundings
inside a tile's products and one per tile at that magnitude."""
import math

import pytest
import torch

from oracle import oracle
from quant_flash_attn_amd.synthetic import make_inputs

DEV = "cuda:0"
OUT_ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 0.0}


def _check(qfa, B, H, Nq, Nk, D, causal, dtype, sdtype, dist="offset", seed=0, layout="bhnd"):
    q, k, v, _ = make_inputs(dist, B, H, max(Nq, Nk), D, seed=seed, dtype=torch.float32)
    q, k, v = q[:, :, :Nq].to(dtype), k[:, :, :Nk].contiguous(), v[:, :, :Nk].contiguous()
    sm = 1.0 / math.sqrt(D)
    kq = tuple(t.to(DEV) for t in (lambda c, s, z, r: (c, s.to(sdtype), z))(*oracle.quantize_per_token_c(k)))
    vq = tuple(t.to(DEV) for t in (lambda c, s, z, r: (c, s.to(sdtype), z))(*oracle.quantize_per_token_c(v)))
    qd = q.to(DEV)
    if layout == "bnhd":   # token-major storage handed over as a permuted view
        turn = lambda t: t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)   # noqa: E731
        qd, kq, vq = turn(qd), (turn(kq[0]),) + kq[1:], (turn(vq[0]),) + vq[1:]
    none = torch.empty(0, dtype=dtype, device=DEV)
    with torch.no_grad():
        o = qfa.quant_flash_attn_quantized_kv(qd, none, none, kq, vq, causal, sm).cpu()
    assert o.dtype == dtype and o.shape == q.shape
    qc, qs, qz, _ = oracle.quantize_per_token_c(q)
    f64 = lambda c, s, z: oracle.dequantize_per_token(c.cpu(), s.cpu(), z.cpu(), torch.float64)   # noqa: E731
    qh, kh, vh = f64(qc, qs, qz), f64(*kq), f64(*vq)
    want, _ = oracle.attn_fwd(qh, kh, vh, causal, sm)
    size, _ = oracle.attn_fwd(qh, kh, vh.abs(), causal, sm)
    offset = (32 + Nk / 32) * 2.0 ** -24 * (1152 + 255) * vq[1].float().max().item()
    err, bound = (o.double() - want).abs(), OUT_ULP[dtype] * want.abs() + 2.0 ** -10 * size + offset
    worst = (err - bound).max().item()
    assert worst <= 0, f"over the bound by {worst:.3e} (largest error {err.max().item():.3e})"


# edges of a 32-key tile and of the deal to four waves; one to four query blocks of 16, ragged
@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("Nq,Nk", [(1, 1), (1, 31), (1, 32), (1, 33), (1, 129), (3, 64), (15, 257), (16, 16), (17, 100), (33, 300),
                                   (64, 130)])
@pytest.mark.parametrize("causal", [True, False])
def test_shapes(qfa, D, Nq, Nk, causal):
    _check(qfa, 1, 2, Nq, Nk, D, causal, torch.bfloat16, torch.float16, seed=Nk)


# keys split over workgroups (few heads, long cache), ragged splits, and no split (many heads)
@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Nq,Nk,D", [(1, 1, 1, 8192, 128), (1, 3, 1, 5001, 64), (1, 2, 5, 3333, 256), (2, 5, 40, 2047, 128),
                                         (9, 64, 1, 70, 128), (9, 61, 2, 300, 64),
                                         # more splits than fill the slots once (5, 3 for none), none where 2 or 3 would
                                         (1, 300, 1, 8192, 128), (2, 170, 1, 4099, 256), (1, 150, 16, 700, 128),
                                         (1, 256, 16, 777, 64)])
def test_splits(qfa, B, H, Nq, Nk, D):
    _check(qfa, B, H, Nq, Nk, D, True, torch.bfloat16, torch.float16, seed=1)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("sdtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("layout", ["bhnd", "bnhd"])
def test_types_and_layouts(qfa, dtype, sdtype, layout):
    for D in (64, 128, 256):
        _check(qfa, 2, 3, 5, 700, D, True, dtype, sdtype, dist="uniform", seed=2, layout=layout)


# either side of the lines between this kernel and the long-query path (keys / head_dim, and one round of workgroups)
@pytest.mark.gpu
@pytest.mark.parametrize("D,H,Nk,edges", [(64, 200, 120, (48, 49)), (64, 200, 128, (64, 65)), (128, 160, 512, (80, 81)),
                                          (64, 120, 512, (112, 113)), (128, 2, 300, (128, 129))])
def test_longest_query_block(qfa, D, H, Nk, edges):
    for Nq in edges:
        _check(qfa, 1, H, Nq, Nk, D, True, torch.float16, torch.float16, dist="normal", seed=Nq)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("Nq", [1, 64, 200])
def test_with_and_without_a_gradient(qfa, Nq, dtype):
    q, k, v, _ = (t.to(DEV) for t in make_inputs("offset", 1, 2, 512, 128, seed=Nq, dtype=dtype))
    q = q[:, :, :Nq].contiguous()
    kq, vq = qfa.asymmetric_quant_per_token(k), qfa.asymmetric_quant_per_token(v)
    with torch.no_grad():
        first = qfa.quant_flash_attn_quantized_kv(q, k, v, kq, vq, True, 0.1)
    again = qfa.quant_flash_attn_quantized_kv(q.requires_grad_(True), k.requires_grad_(True), v, kq, vq, True, 0.1)
    assert torch.equal(again.detach(), first)
    again.sum().backward()
    assert torch.isfinite(q.grad).all() and torch.isfinite(k.grad).all()


@pytest.mark.gpu
def test_growing_scores_and_one_sided_rows(qfa):
    """Scores that grow along the keys move the running maximum in every tile; all-positive rows pin the zero points."""
    for D in (64, 128, 256):
        g = torch.Generator().manual_seed(D)
        q = torch.rand(1, 2, 3, D, generator=g).to(torch.float16)
        k = torch.rand(1, 2, 900, D, generator=g) * torch.linspace(0.1, 8.0, 900).view(1, 1, -1, 1)
        kq = tuple(t.to(DEV) for t in oracle.quantize_per_token_c(k)[:3])
        none = torch.empty(0, dtype=torch.float16, device=DEV)
        with torch.no_grad():
            o = qfa.quant_flash_attn_quantized_kv(q.to(DEV), none, none, kq, kq, True, 0.5).cpu()
        qh = oracle.dequantize_per_token(*oracle.quantize_per_token_c(q)[:3], torch.float64)
        kh = oracle.dequantize_per_token(*(t.cpu() for t in kq), torch.float64)
        want, _ = oracle.attn_fwd(qh, kh, kh, True, 0.5)
        # scores reach 0.5 * sum_d q k ~ 8 D: their fp32 rounding is 2^-23 of that in the exponent
        offset = (32 + 900 / 32) * 2.0 ** -24 * (1152 + 255) * kq[1].max().item()
        bound = (2.0 ** -11 + 2.0 ** -10 + 8 * D * 2.0 ** -22) * want.abs() + offset
        assert ((o.double() - want).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("dtype,sdtype,size", [
    (torch.bfloat16, torch.float16, 1.0), (torch.bfloat16, torch.float16, 1e-2), (torch.bfloat16, torch.float16, 1e-4),
    (torch.float16, torch.float16, 1e-3), (torch.float32, torch.float16, 1e-4), (torch.bfloat16, torch.float16, 1e6),
    (torch.bfloat16, torch.float32, 1e-20), (torch.bfloat16, torch.bfloat16, 1e20), (torch.bfloat16, torch.float32, "ramp"),
    (torch.bfloat16, torch.float32, "masked out"), (torch.float32, torch.float32, "rising scores")])
def test_size_of_the_values(qfa, D, dtype, sdtype, size):
    """V of any size, alike for all keys or not: values that grow by 2^40 along the keys, large values at keys that hardly
    any query attends to, and scores that rise (by hundreds) while the values fall.

    Bound: as above, but every term is weighted with the probabilities (the scales differ by key), and binary16's smallest
    step, 2^-24, is one of the largest p_j scale_j of the row, once per key, times |code - zero point| <= 255."""
    B, H, Nq, Nk = 1, 3, 5, 2100
    q, k, v, _ = make_inputs("normal", B, H, Nk, D, seed=D, dtype=torch.float32)
    q, sm = q[:, :, :Nq].to(dtype), 1.0 / math.sqrt(D)
    ramp = torch.arange(Nk).view(1, 1, -1, 1) / Nk
    if size == "ramp":
        v = v * 2.0 ** (40 * ramp - 20)
    elif size == "masked out":     # scores near -40 at the keys with large values, in the first tile and later
        q = (q.float().abs() + 0.5).to(dtype)
        far = (ramp < 0.01) | ((ramp > 0.5) & (ramp < 0.52))
        k = torch.where(far, -40 * sm * torch.ones_like(k), k * 0.1)
        v = torch.where(far, v * 1e5, v)
    elif size == "rising scores":
        q = (q.float().abs() + 0.5).to(dtype)
        k, v = k * 0.1 + 40 * ramp, v * 2.0 ** (-60 * ramp)
    else:
        v = v * size
    kq = tuple(t.to(DEV) for t in oracle.quantize_per_token_c(k)[:3])
    vc, vs, vz, _ = oracle.quantize_per_token_c(v)
    kq = (kq[0], kq[1].to(sdtype), kq[2])
    vq = (vc.to(DEV), vs.to(sdtype).to(DEV), vz.to(DEV))
    none = torch.empty(0, dtype=dtype, device=DEV)
    with torch.no_grad():
        o = qfa.quant_flash_attn_quantized_kv(q.to(DEV), none, none, kq, vq, True, sm).cpu()
    f64 = lambda c, s, z: oracle.dequantize_per_token(c.cpu(), s.cpu(), z.cpu(), torch.float64)   # noqa: E731
    qh, kh, vh = f64(*oracle.quantize_per_token_c(q)[:3]), f64(*kq), f64(*vq)
    want, lse = oracle.attn_fwd(qh, kh, vh, True, sm)
    s = (qh @ kh.transpose(-1, -2)) * sm
    seen = torch.arange(Nk) <= torch.arange(Nq).view(-1, 1) + Nk - Nq
    p = torch.where(seen, torch.exp(s - lse[..., None]), torch.zeros(()).double())
    ps = p * vq[1].cpu().double().reshape(B, H, 1, Nk)
    size_of = p @ vh.abs()
    # (fp32 scores: a rounding of the largest |score| in the exponent, twice)
    bound = (OUT_ULP[dtype] * want.abs() + (2.0 ** -10 + 2.0 ** -22 * float(s.abs().max())) * size_of
             + ((32 + Nk / 32) * 2.0 ** -24 * (1152 + 255) * ps.sum(-1, keepdim=True))
             + Nk * 255 * 2.0 ** -25 * ps.max(-1, keepdim=True).values)
    if dtype == torch.float16:
        bound = bound + 2.0 ** -25
    excess = (o.double() - want).abs() - bound
    assert torch.isfinite(o.float()).all() and excess.max() <= 0, (
        f"over the bound by {(excess / bound).max().item():.2f} times it; relative error "
        f"{float((o.double() - want).norm() / want.norm()):.2e}")


@pytest.mark.gpu
def test_graph_capture_and_replay(qfa):
    q, k, v, _ = (t.to(DEV) for t in make_inputs("offset", 1, 4, 4096, 128, seed=3))
    q = q[:, :, :1].contiguous()
    kq, vq = qfa.asymmetric_quant_per_token(k), qfa.asymmetric_quant_per_token(v)
    none = torch.empty(0, dtype=q.dtype, device=DEV)
    run = lambda: qfa.quant_flash_attn_quantized_kv(q, none, none, kq, vq, True, 0.1)   # noqa: E731
    with torch.no_grad():
        want = run().clone()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = run()
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
            run()
            torch.cuda.synchronize()


def test_argument_errors_need_no_gpu(qfa):
    from quant_flash_attn_amd import _lib
    L, p = _lib.lib(), 0x1000   # never dereferenced: validation fails first

    def call(q=p, qdt=2, sdt=1, Nq=1, Nk=64, D=128, sm=0.1, causal=1, skn=None, ws=None, ws_bytes=0):
        sq, sk = (Nq * D, Nq * D, D), (Nk * (skn or D), Nk * (skn or D), skn or D)
        return L.qfa_attn_fwd_cache(q, qdt, p, p, p, p, p, p, sdt, p, 1, 1, Nq, Nk, D, *sq, *sk, *sk, *sq, sm, causal, ws,
                                    ws_bytes, None)
    assert call(q=None) == -1 and b"null" in L.qfa_last_error()
    assert call(qdt=7) == -1 and b"q_dtype" in L.qfa_last_error()
    assert call(sdt=7) == -1 and b"scale_dtype" in L.qfa_last_error()
    assert call(D=96) == -2 and b"head_dim" in L.qfa_last_error()
    assert call(Nq=65) == -2 and b"causal" in L.qfa_last_error()
    assert call(sm=0.0) == -1 and b"sm_scale" in L.qfa_last_error()
    assert call(q=p + 2) == -1 and b"aligned" in L.qfa_last_error()
    assert call(skn=1 << 23) == -2 and b"token strides" in L.qfa_last_error()
    assert call(Nk=8192, ws=p, ws_bytes=8) == -1 and b"workspace" in L.qfa_last_error()
    assert L.qfa_attn_fwd_cache_workspace_bytes(8, 32, 1, 8192, 128) > 0
    assert L.qfa_attn_fwd_cache_workspace_bytes(64, 32, 1, 8192, 128) == 0
