"""bf16 Q and O of the shared-KV backward are cast by the launch that scales dO: the same gradients whatever way they are cast."""
import pytest
import torch

from quant_flash_attn_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("B,H,Nq,D", [(1, 1, 1, 64), (1, 3, 5, 256), (2, 3, 17, 128), (3, 5, 100, 64)])
def test_cast_beside_the_scaling(qfa, B, H, Nq, D):
    L, n = _lib.lib(), B * H * Nq * D
    g = torch.Generator().manual_seed(n)
    do, x0, x1 = (torch.randn(n, generator=g).mul(s).bfloat16().to(DEV) for s in (1e-3, 1.0, 1e-6))   # (subnormal in binary16)
    x0[0] = 1e6   # beyond binary16
    scale = torch.rand(1001, generator=g).to(DEV)
    ws = torch.empty(L.qfa_dout_normalise_workspace_bytes(), dtype=torch.uint8, device=DEV)
    new = lambda: torch.full((n + 8,), 7.0, dtype=torch.float16, device=DEV)
    a, b, y0, y1 = new(), new(), new(), new()
    back = torch.empty(2, device=DEV)
    st = torch.cuda.current_stream().cuda_stream
    args = lambda out, i: (do.data_ptr(), 2, n, scale.data_ptr(), 0, 1001, ws.data_ptr(), out.data_ptr(), back[i:].data_ptr())
    assert L.qfa_dout_normalise(*args(a, 0), st) == 0
    assert L.qfa_dout_normalise_cast(*args(b, 1), x0.data_ptr(), y0.data_ptr(), x1.data_ptr(), y1.data_ptr(), st) == 0
    assert torch.equal(a, b) and back[0] == back[1]
    assert torch.equal(y0[:n], x0.half()) and torch.equal(y1[:n], x1.half())
    assert all((t[n:] == 7.0).all() for t in (a, b, y0, y1))
    assert L.qfa_dout_normalise_cast(*args(b, 1), None, None, x1.data_ptr(), y1.data_ptr(), st) == -1
    assert L.qfa_dout_normalise_cast(*args(b, 1), x0.data_ptr(), None, None, None, st) == -1


@pytest.mark.parametrize("Nq,D,direct", [(20, 128, 1), (128, 128, 1), (129, 128, 0), (150, 64, 0), (17, 256, 0), (100, 256, 0)])
def test_strided_queries_give_the_same_gradients(qfa, Nq, D, direct):
    """Blocks whose rows a workgroup does not hold are cast in front of the backward: contiguous ones by the launch that scales dO,
    strided ones by a copy of their own.  Shorter ones are cast inside the kernels (direct), from whatever strides."""
    assert _lib.lib().qfa_attn_bwd_shared_kv_is_direct(Nq, D) == direct
    B, H, Nk, sm = 2, 3, 300, 0.09
    g = torch.Generator().manual_seed(2)
    q0 = torch.randn((B, Nq, H, D), generator=g).bfloat16().to(DEV).transpose(1, 2)
    kv = torch.randn((B, H, Nk, D), generator=g).bfloat16().to(DEV)
    do = torch.randn((B, H, Nq, D), generator=g).bfloat16().to(DEV)
    quant = qfa.asymmetric_quant_per_token(kv)
    res = []
    for q in (q0, q0.contiguous()):
        leaves = [q.detach().requires_grad_(True), kv.detach().requires_grad_(True)]
        assert leaves[0].is_contiguous() == (q is not q0)
        res.append(torch.autograd.grad(qfa.quant_flash_attn(leaves[0], leaves[1], quant, sm), leaves, do))
    assert all(torch.equal(a, b) for a, b in zip(*res))
