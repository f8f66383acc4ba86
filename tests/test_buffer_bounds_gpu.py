"""What the kernels rely on where rows, keys or whole tiles do not exist: a load through a buffer descriptor returns zeros from the
descriptor's end on, and the scalar offset of the load counts -- also where it alone lies past the end, and with an empty descriptor.
(The compiler's documentation leaves the scalar offset out of the check.)  Every load here stays inside one allocation, so a
load that was not stopped would show as the words that lie there."""
import ctypes
import math
import os
import subprocess

import pytest
import torch

from quant_flash_attn_amd import build

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native")
LIB = os.path.join(HERE, "libbuffer_bounds.so")
BYTES = 1 << 16
WIDTH = [16, 16, 8, 4, 2, 1]   # bytes of the loads: straight to LDS, then into registers


@pytest.fixture(scope="module")
def load():
    if not os.path.exists(LIB):
        subprocess.run([build._hipcc(), *build.COMMON, "-shared", "-x", "hip", os.path.join(HERE, "buffer_bounds.hip"), "-o", LIB],
                       check=True, capture_output=True)
    f = ctypes.CDLL(LIB).load_through_descriptor
    f.argtypes = [ctypes.c_void_p, ctypes.c_uint, ctypes.c_uint, ctypes.c_uint, ctypes.c_void_p, ctypes.c_void_p]
    return f


@pytest.mark.gpu
@pytest.mark.parametrize("records", [0, 16, 512, 1024, 4096, 8208])
@pytest.mark.parametrize("soffset", [0, 16, 32, 1024, 4096, 8192, 32768])
def test_loads_end_with_their_descriptor(load, records, soffset):
    base = (torch.arange(BYTES // 4, dtype=torch.int32) | 0x5a000000).to("cuda:0")
    out = torch.full((6, 64, 4), -1, dtype=torch.int32, device="cuda:0")
    assert load(base.data_ptr(), BYTES, records, soffset, out.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    got, words = out.cpu(), base.cpu()[soffset // 4:soffset // 4 + 256].reshape(64, 4)
    inside = soffset + 16 * torch.arange(64) < records   # (a multiple of 16: no load is cut)
    for i, width in enumerate(WIDTH):
        want = words.clone()
        want[:, (width + 3) // 4:] = 0
        if width < 4:
            want[:, 0] &= (1 << 8 * width) - 1
        want[~inside] = 0
        assert torch.equal(got[i], want), (width, i)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("Nq", [33, 49, 63])
def test_rows_of_the_next_head_stay_out_shared_kv(qfa, Nq, D):
    """Every row of a head's Q and dO is infinite: the blocks of 32 rows that end the head in front of it have the bits that they have
    without."""
    BH, Nk, h, sm = 5, 100, 2, 1.0 / math.sqrt(D)
    g = torch.Generator().manual_seed(Nq)
    kv, q, do = (torch.randn((1, BH, n, D), generator=g).to(torch.float16).to("cuda:0") for n in (Nk, Nq, Nq))
    quant = qfa.asymmetric_quant_per_token(kv)

    def run(q, do):
        o, lse = qfa.attn_fwd_shared_kv(q, *quant, sm)
        return o, *qfa.attn_bwd_shared_kv(q, *quant, o, do, lse, sm)
    want = run(q, do)
    q, do = q.clone(), do.clone()
    q[:, h + 1] = do[:, h + 1] = float("inf")
    others = [i for i in range(BH) if i != h + 1]
    for a, b in zip(run(q, do), want):
        assert torch.isfinite(b).all() and torch.equal(a[:, others], b[:, others])


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("N", [33, 49, 63, 97])
def test_rows_of_the_next_head_stay_out(qfa, N, causal, D):
    """The same for V and dO of the INT8-score path."""
    BH, h, sm = 5, 2, 1.0 / math.sqrt(D)
    g = torch.Generator().manual_seed(N)
    q, k, v, do = (torch.randn((1, BH, N, D), generator=g).to(torch.bfloat16).to("cuda:0") for _ in range(4))

    def run(v, do):
        leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
        o = qfa.quant_flash_attn_qkv(*leaves, causal, sm)
        return o.detach(), *torch.autograd.grad(o, leaves, do)
    want = run(v, do)
    others = [i for i in range(BH) if i != h + 1]
    for which in (0, 1):
        args = [v.clone(), do.clone()]
        args[which][:, h + 1] = float("inf")
        for a, b in zip(run(*args), want):
            assert torch.isfinite(b).all() and torch.equal(a[:, others], b[:, others])
