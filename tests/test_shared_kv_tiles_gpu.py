"""The shared-KV kernels that expand a tile of keys once per workgroup (forward, dQ), the dKV kernel with resident rows, and
the backward with its keys split over workgroups, at the sizes where they can go wrong (the backward of 33 to 128 queries in one
pass has tests of its own; cases here are on both sides of its line): one key, tiles and blocks of 32, 64
and 128 with one more or one less, two and four waves side by side, one wave without queries, and few heads (splits).
Many heads make the dispatch take these kernels at small sizes; the first, a middle and the last head are compared with the
oracle, with the tolerances of helpers.py."""
import math
import random

import pytest
import torch

from helpers import COS_TOL, assert_close, max_abs
from oracle import oracle
from plans import skv_pass_takes, skv_tile_dq_plan, skv_tile_fwd_plan
from quant_flash_attn_amd import _lib

DEV = "cuda:0"

# the kernels that forward and backward (dQ) of a case are to reach, at head_dim 64, 128 and 256
TILES = ["tiles, tiles"] * 3
PASS = ["tiles, pass per head"] * 2 + TILES[:1]
CASES = [
    # heads, Nq, Nk, dtype, scale dtype, kernels
    (512, 33, 1, torch.float16, torch.float16, ["16 queries, pass per head", "tiles, pass per head", "16 queries, 16 queries"]),   # one key
    (512, 65, 1, torch.float16, torch.float16, PASS),
    (512, 65, 31, torch.float16, torch.float32, PASS),     # three blocks on four waves, one key less than a block
    (300, 200, 33, torch.bfloat16, torch.float16, TILES),   # two workgroups per head, four and three blocks
    (256, 97, 65, torch.float16, torch.float16, TILES[:1] + PASS[1:]),     # one key more than a tile; resident rows, the last block one query
    (256, 128, 129, torch.float16, torch.float16, TILES[:1] + PASS[1:]),   # all resident rows, one key more than four waves' tiles
    (256, 129, 128, torch.bfloat16, torch.float32, TILES),  # one query more than the resident rows
    (64, 512, 97, torch.float16, torch.float16, TILES),
    (600, 64, 70, torch.float16, torch.bfloat16, PASS[:2] + ["16 queries, 16 queries"]),
    # the two kernels beside the line of the pass: 257 to 319 heads of 64, more than 1024 heads of 128 with two tiles of keys at most
    (270, 64, 1, torch.bfloat16, torch.float32, ["16 queries, tiles"] + ["16 queries, 16 queries"] * 2),
    (270, 65, 31, torch.float16, torch.float16, ["16 queries, tiles", "tiles, 16 queries", "16 queries, 16 queries"]),
    (300, 64, 70, torch.bfloat16, torch.float16, ["16 queries, tiles", "16 queries, pass per head", "16 queries, 16 queries"]),
    (270, 97, 65, torch.float16, torch.float16, TILES),
    (280, 128, 129, torch.float16, torch.float32, TILES),
    (1100, 64, 1, torch.float16, torch.float16, PASS[:1] + ["tiles, tiles", "16 queries, tiles"]),
    (1100, 97, 31, torch.bfloat16, torch.float32, PASS[:1] + TILES[1:]),
    (1100, 128, 65, torch.float16, torch.float16, PASS[:1] + TILES[1:]),
    (1100, 65, 128, torch.bfloat16, torch.float16, PASS[:1] + TILES[1:]),
    (40, 100, 2001, torch.float16, torch.float16, ["tiles split, 16 queries"] * 3),
    (40, 65, 5001, torch.bfloat16, torch.float16, ["tiles split, tiles split"] * 2 + ["tiles split, 16 queries"]),
    (600, 32, 70, torch.float16, torch.float16, ["16 queries, one pass"] * 2 + ["16 queries, 16 queries"]),
    (3, 16, 3001, torch.float16, torch.float16, ["16 queries split, one pass split"] * 3),
    (2, 31, 2500, torch.bfloat16, torch.float32, ["16 queries split, one pass split"] * 2 + ["16 queries split, tiles split"]),
    (1, 200, 9001, torch.float16, torch.float16, ["16 queries split, tiles split"] * 3),
]


def _kernels(BH, Nq, Nk, D):
    L, fwd, dq = _lib.lib(), skv_tile_fwd_plan(BH, Nq, Nk, D), skv_tile_dq_plan(BH, Nq, Nk, D)
    parts = [f(1, BH, Nq, Nk, D) for f in (L.qfa_attn_fwd_shared_kv_workspace_bytes, L.qfa_attn_bwd_shared_kv_workspace_bytes)]
    names = ["tiles" if fwd.waves else "16 queries",
             "one pass" if Nq <= (16 if D == 256 else 32) else "pass per head" if skv_pass_takes(BH, Nq, Nk, D) else
             "tiles" if dq.waves else "16 queries"]
    return ", ".join(n + (" split" if p else "") for n, p in zip(names, parts))


def test_cases_reach_the_kernels_they_name(qfa):
    for BH, Nq, Nk, _, _, kernels in CASES:
        assert [_kernels(BH, Nq, Nk, D) for D in (64, 128, 256)] == kernels, (BH, Nq, Nk)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("BH,Nq,Nk,dtype,sdtype", [c[:5] for c in CASES])
def test_tiles_vs_oracle(qfa, BH, Nq, Nk, dtype, sdtype, D):
    g = torch.Generator().manual_seed(BH + Nq + Nk + D)
    kv = (torch.randn((1, BH, Nk, D), generator=g) + 0.3 * torch.randn((1, BH, Nk, 1), generator=g)).to(dtype)
    q, do = (torch.randn((1, BH, Nq, D), generator=g).to(dtype) for _ in range(2))
    sm = 1.0 / math.sqrt(D)
    qd, kvd = q.to(DEV).requires_grad_(True), kv.to(DEV).requires_grad_(True)
    codes, scale, zp = qfa.asymmetric_quant_per_token(kvd.detach(), scale_dtype=sdtype)
    o = qfa.quant_flash_attn(qd, kvd, (codes, scale, zp), sm)
    dq, dkv = torch.autograd.grad(o, [qd, kvd], do.to(DEV))
    o2, lse = qfa.attn_fwd_shared_kv(qd.detach(), codes, scale, zp, sm)
    torch.cuda.synchronize()
    assert torch.equal(o, o2)
    pick = sorted({0, BH // 2, BH - 1})
    q, do, codes, scale, zp, o, lse, dq, dkv = (t.detach()[:, pick].cpu() for t in (q, do, codes, scale, zp, o, lse, dq, dkv))
    o_ref, lse_ref = oracle.legacy_fwd(q, codes, scale, zp, sm)
    assert_close("O", o, o_ref, scaled=True)
    assert max_abs(lse, lse_ref) < 2.0 ** -8
    (dq_ref, dkv_ref), (nq, nkv) = oracle.legacy_bwd(q, codes, scale, zp, do, sm, o=o, spread=True)
    assert_close("dQ", dq, dq_ref, scaled=True, spread=nq, cos_tol=COS_TOL if Nk > 1 else -1.0)   # one key: dQ is zero
    assert_close("dKV", dkv, dkv_ref, scaled=True, spread=nkv)


@pytest.mark.gpu
@pytest.mark.parametrize("D,BH,whole", [(64, 512, True), (64, 300, False), (128, 512, True), (128, 1100, False), (256, 512, False)])
def test_infinite_rows_stay_with_their_queries(qfa, D, BH, whole):
    """An infinite query or dO row reaches O and dQ of its own query only.  The others may be taken against another reference
    maximum (a wave moves its queries' references together), which rounds their probabilities differently: 2^-11 each, so
    2^-9 of the largest value bounds what two roundings of a weighted sum and of the result can move."""
    Nq, Nk = 65, 70
    assert _kernels(BH, Nq, Nk, D).split(", ")[1] == ("pass per head" if whole else "tiles")
    g = torch.Generator().manual_seed(D)
    kv, q, do = (torch.randn(s, generator=g).to(torch.float16).to(DEV) for s in ((1, BH, Nk, D), (1, BH, Nq, D), (1, BH, Nq, D)))
    codes, scale, zp = qfa.asymmetric_quant_per_token(kv)
    sm = 1.0 / math.sqrt(D)

    def run(q, do):
        o, lse = qfa.attn_fwd_shared_kv(q, codes, scale, zp, sm)
        return o, qfa.attn_bwd_shared_kv(q, codes, scale, zp, o, do, lse, sm)[0]
    want = run(q, do)
    q2, do2 = q.clone(), do.clone()
    q2[:, :, 40, 3] = float("inf")
    do2[:, :, 7] = float("inf")
    got = run(q2, do2)
    keep = [i for i in range(Nq) if i not in (7, 40)]
    for a, b in zip(got, want):
        a, b = a[:, :, keep].float(), b[:, :, keep].float()
        assert torch.isfinite(a).all()
        assert float((a - b).abs().max()) <= 2.0 ** -9 * float(b.abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("sm", [1e-25, 1e-3, 30.0])
def test_softmax_scales(qfa, sm):
    """The forward multiplies the key scales by sm_scale: O and LSE at scales far from 1/sqrt(D)."""
    BH, Nq, Nk, D = 512, 65, 130, 128
    g = torch.Generator().manual_seed(3)
    kv, q = (torch.randn(s, generator=g).to(torch.float16) for s in ((1, BH, Nk, D), (1, BH, Nq, D)))
    codes, scale, zp = qfa.asymmetric_quant_per_token(kv.to(DEV))
    o, lse = (t[:, :2].cpu() for t in qfa.attn_fwd_shared_kv(q.to(DEV), codes, scale, zp, sm))
    o_ref, lse_ref = oracle.legacy_fwd(q[:, :2], *(t[:, :2].cpu() for t in (codes, scale, zp)), sm)
    assert_close("O", o, o_ref, scaled=True)
    # scores reach 30 * 60: binary32 of the exponent in log2 units loses 2^-24 of that per operation
    assert max_abs(lse, lse_ref) < 2.0 ** -8 * max(1.0, float(lse_ref.abs().max()) * 2.0 ** -8)


def test_backward_workspace_is_bounded(qfa):
    """Partial results of a split stay within 64 MiB, and a chip that is full is not split (head_dim up to 128)."""
    L, rng = _lib.lib(), random.Random(2)
    for _ in range(20000):
        B, H, Nq, Nk = rng.randint(1, 64), rng.randint(1, 64), rng.choice((1, 16, 17, 32, 33, 512, 2000)), rng.randint(1, 40000)
        for D in (64, 128, 256):
            assert 0 <= L.qfa_attn_bwd_shared_kv_workspace_bytes(B, H, Nq, Nk, D) <= (64 << 20)
    assert L.qfa_attn_bwd_shared_kv_workspace_bytes(512, 16, 16, 3000, 128) == 0
