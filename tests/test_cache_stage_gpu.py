"""The pass over an INT8 K / V cache in front of the INT8-score forward: whole numbers and 16-bit values as the separate passes
give them, at the edges of a workgroup's tokens (128, 64, 32 at head_dim 64, 128, 256)."""
import pytest
import torch

from quant_flash_attn_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CODE = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("N", [1, 31, 32, 129, 1000])
@pytest.mark.parametrize("ks,vs,out", [(torch.float16, torch.float16, torch.bfloat16), (torch.bfloat16, torch.float32, torch.float16),
                                       (torch.float32, torch.bfloat16, torch.bfloat16)])
def test_cache_stage(qfa, D, N, ks, vs, out):
    B, H = 2, 3
    g = torch.Generator().manual_seed(N + D)
    code = lambda: torch.randint(-128, 128, (B, N, H, D), dtype=torch.int8, generator=g).to(DEV).transpose(1, 2)   # [B,N,H,D] storage
    k, v = code(), code().contiguous()
    sk, sv = (torch.rand((B, H, N, 1), generator=g).mul(0.1).to(dt).to(DEV) for dt in (ks, vs))
    zv = torch.randint(-128, 128, (B, H, N, 1), dtype=torch.int8, generator=g).to(DEV)
    guard = lambda n, dt: torch.full((n + 64,), 7, dtype=dt, device=DEV)
    widen = ks != torch.float32
    rowsum, k32, v16 = guard(B * H * N, torch.int32), guard(B * H * N, torch.float32), guard(B * H * N * D, out)
    rc = _lib.lib().qfa_cache_stage(k.data_ptr(), sk.data_ptr(), CODE[ks], k32.data_ptr() if widen else None, rowsum.data_ptr(),
                                    v.data_ptr(), sv.data_ptr(), CODE[vs], zv.data_ptr(), v16.data_ptr(), CODE[out], B, H, N, D,
                                    *k.stride()[:3], *v.stride()[:3], torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.lib().qfa_last_error()
    n = B * H * N
    assert torch.equal(rowsum[:n], k.sum(-1, dtype=torch.int32).flatten())
    if widen:
        assert torch.equal(k32[:n], sk.float().flatten())
    assert torch.equal(v16[:n * D].view(B, H, N, D), _lib.host().dequant(v, sv, zv, out))
    for t, m in ((rowsum, n), (v16, n * D)):
        assert (t[m:] == 7).all()
    assert _lib.lib().qfa_cache_stage(k.data_ptr(), sk.data_ptr(), CODE[ks], None, rowsum.data_ptr(), v.data_ptr(), sv.data_ptr(), 5,
                                      zv.data_ptr(), v16.data_ptr(), CODE[out], B, H, N, D, *k.stride()[:3], *v.stride()[:3], None) == -1


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("Nq,N", [(1, 33), (32, 1), (33, 32), (129, 1000), (257, 31)])
@pytest.mark.parametrize("dtype,out", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16), (torch.float32, torch.bfloat16)])
def test_cache_stage_with_queries(qfa, D, Nq, N, dtype, out):
    """The queries' codes, scales, zero points and row sums are those of the quantizer's own launch, and the cache's are those without
    queries."""
    B, H, L = 2, 3, _lib.lib()
    g = torch.Generator().manual_seed(N + D + Nq)
    q = torch.randn((B, Nq, H, D), generator=g).to(dtype).to(DEV).transpose(1, 2)   # [B,N,H,D] storage
    k, v = (torch.randint(-128, 128, (B, H, N, D), dtype=torch.int8, generator=g).to(DEV) for _ in range(2))
    sk, sv = (torch.rand((B, H, N, 1), generator=g).mul(0.1).half().to(DEV) for _ in range(2))
    zv = torch.randint(-128, 128, (B, H, N, 1), dtype=torch.int8, generator=g).to(DEV)
    full = lambda n, dt: torch.full((n + 64,), 7, dtype=dt, device=DEV)
    nq, n = B * H * Nq, B * H * N
    cache = lambda: (full(n, torch.float32), full(n, torch.int32), full(n * D, out))
    (k32, ksum, v16), (k32_, ksum_, v16_) = cache(), cache()
    qo = codes, scale, zp, qsum = full(nq * D, torch.int8), full(nq, torch.float32), full(nq, torch.int8), full(nq, torch.int32)
    rest = lambda a, b, c: (k.data_ptr(), sk.data_ptr(), 1, a.data_ptr(), b.data_ptr(), v.data_ptr(), sv.data_ptr(), 1, zv.data_ptr(),
                            c.data_ptr(), CODE[out], B, H, N, D, *k.stride()[:3], *v.stride()[:3], torch.cuda.current_stream().cuda_stream)
    queries = lambda code: (q.data_ptr(), code, *(t.data_ptr() for t in qo), Nq, *q.stride()[:3], H * Nq * D, Nq * D, D)
    assert L.qfa_cache_stage_q(*queries(CODE[dtype]), *rest(k32, ksum, v16)) == 0, L.qfa_last_error()
    assert L.qfa_cache_stage(*rest(k32_, ksum_, v16_)) == 0, L.qfa_last_error()
    want = qfa.quantize_for_attention(q)
    for got, ref, m in zip(qo, (want.codes, want.scale, want.zero_point, want.rowsum), (nq * D, nq, nq, nq)):
        assert torch.equal(got[:m], ref.flatten()) and (got[m:] == 7).all()
    assert torch.equal(k32, k32_) and torch.equal(ksum, ksum_) and torch.equal(v16, v16_)
    other = torch.float16 if out == torch.bfloat16 else torch.bfloat16
    assert L.qfa_cache_stage_q(*queries(CODE[other]), *rest(k32, ksum, v16)) == -1
