"""The shared-KV backward in one pass of 33 to 128 queries (one workgroup per head, where there are enough heads), at the sizes where
it can go wrong: one key, blocks of 32 and tiles of 64 keys with one more or one less, odd and even numbers of tiles, one to five of
them (its rings of tiles hold four and five), blocks of 32 queries that hold one or none, a partly filled second half of the queries'
waves, strides."""
import math

import pytest
import torch

from helpers import COS_TOL, assert_close
from oracle import oracle
from plans import skv_pass_takes, skv_pass_takes_unsplit, skv_tile_dq_plan
from quant_flash_attn_amd import _lib

DEV = "cuda:0"
NQ = [33, 61, 64, 65, 96, 97, 128]
NK = [1, 31, 63, 64, 65, 97, 128, 129, 191, 256, 300, 389]
HEADS = {64: 320, 128: 128}   # the fewest


def test_line(qfa):
    """Which calls take it, and that they need no scratch."""
    for D, least in HEADS.items():
        for Nq in (32, 33, 128, 129):
            for BH in (least - 1, least, 5000):
                takes = 33 <= Nq <= 128 and BH >= least
                assert bool(skv_pass_takes(BH, Nq, 500, D)) == takes
                if takes:
                    assert _lib.lib().qfa_attn_bwd_shared_kv_workspace_bytes(1, BH, Nq, 500, D) == 0
    assert not skv_pass_takes(5000, 64, 500, 256)
    assert not skv_pass_takes(270, 64, 500, 128) and not skv_pass_takes(5000, 64, 128, 128)


def test_scratch_where_strides_may_not_fit(qfa):
    """Rows of a head further apart than 31-bit offsets reach go to the two kernels, which want scratch to split few heads' keys."""
    for B, H, Nq, Nk, D in [(1, 160, 128, 70000, 128), (2, 128, 100, 70000, 128), (1, 448, 128, 70000, 64)]:
        assert skv_pass_takes(B * H, Nq, Nk, D)
        plan = skv_tile_dq_plan(B * H, Nq, Nk, D)
        want = B * H * Nq * plan.splits * D * 4
        assert plan.splits > 1 and _lib.lib().qfa_attn_bwd_shared_kv_workspace_bytes(B, H, Nq, Nk, D) == want


@pytest.mark.parametrize("BH,Nq,Nk,D,us", [   # us of the one pass and of the two kernels with their splits, on an MI355X
    (320, 72, 16000, 64, (746, 616)), (327, 86, 4558, 64, (216, 204)), (340, 72, 16000, 64, (743, 693)), (320, 40, 2500, 64, (84, 90)),
    (360, 72, 6000, 64, (281, 288)), (384, 96, 16000, 64, (766, 760)), (512, 65, 4000, 64, (194, 253)),
    (513, 40, 16000, 64, (916, 776)), (525, 34, 6365, 64, (377, 325)), (576, 33, 4000, 64, (236, 226)), (513, 65, 1500, 64, (120, 122)),
    (660, 40, 2500, 64, (172, 161)), (660, 72, 4000, 64, (323, 334)), (700, 40, 2500, 64, (171, 174)),
    (128, 65, 16000, 128, (539, 462)), (136, 74, 14424, 128, (486, 479)), (128, 97, 1000, 128, (44, 64)), (160, 65, 16000, 128, (550, 577)),
    (274, 111, 3997, 128, (366, 345)), (288, 65, 8000, 128, (569, 554)), (288, 97, 1000, 128, (88, 113)), (320, 65, 16000, 128, (1100, 1161)),
    (513, 97, 4000, 128, (454, 634)),
    # where edges in heads and keys alone sent blocks that fill their waves the wrong way
    (372, 127, 6309, 64, (311, 367)), (630, 107, 2340, 64, (201, 244)), (641, 104, 2400, 64, (211, 262)), (644, 56, 2350, 64, (146, 181)),
    (133, 59, 4775, 128, (119, 147)), (297, 116, 2560, 128, (210, 290)), (299, 104, 2080, 128, (168, 226))])
def test_choice_is_not_slower(qfa, BH, Nq, Nk, D, us):
    """Few heads, and a few more than fill the chip: whichever way a call goes is not slower than the other by more than the estimates
    of the two are off together: 3 and 5 % rms, 8 %."""
    takes = skv_pass_takes(BH, Nq, Nk, D)
    assert us[0 if takes else 1] <= 1.08 * us[1 if takes else 0]


@pytest.mark.parametrize("BH,Nq,Nk,D,split", [(355, 85, 13075, 64, True), (130, 60, 23096, 128, True), (521, 40, 5877, 64, False),
                                              (270, 100, 8000, 128, False), (300, 100, 8000, 64, False), (512, 129, 8000, 64, False)])
def test_without_scratch(qfa, BH, Nq, Nk, D, split):
    """A call that would go to the two kernels for their split goes to the one pass if it brings no scratch; others do not."""
    assert not skv_pass_takes(BH, Nq, Nk, D) and (Nq > 128 or not split or skv_tile_dq_plan(BH, Nq, Nk, D).splits > 1)
    assert skv_pass_takes_unsplit(BH, Nq, Nk, D) == split
    assert skv_pass_takes_unsplit(BH, 64, 500, D) == skv_pass_takes(BH, 64, 500, D)


@pytest.mark.gpu
def test_with_and_without_scratch(qfa):
    """The autograd entry, which brings scratch, and the public call, which does not, take different kernels: both against the oracle."""
    BH, Nq, Nk, D, sm = 330, 72, 8500, 64, 0.125
    assert not skv_pass_takes(BH, Nq, Nk, D) and skv_pass_takes_unsplit(BH, Nq, Nk, D)
    q, kv, do, qd, kvd, dod = _case(BH, Nq, Nk, D, torch.float16, torch.float16, "heads")
    quant = qfa.asymmetric_quant_per_token(kvd)
    o, lse = qfa.attn_fwd_shared_kv(qd, *quant, sm)
    got = {"public": qfa.attn_bwd_shared_kv(qd, *quant, o, dod, lse, sm)}
    leaves = qd.requires_grad_(True), kvd.requires_grad_(True)
    got["autograd"] = torch.autograd.grad(qfa.quant_flash_attn(*leaves, quant, sm), leaves, dod)
    assert not torch.equal(got["public"][0], got["autograd"][0])
    pick = [0, BH // 2, BH - 1]
    refs, spreads = oracle.legacy_bwd(*(t[:, pick].detach().cpu() for t in (q, *quant, do)), sm, o=o[:, pick].cpu(), spread=True)
    for name, grads in got.items():
        for a, b, n in zip(grads, refs, spreads):
            assert_close(name, a[:, pick].cpu(), b, scaled=True, spread=n)


def _case(BH, Nq, Nk, D, dtype, sdtype, layout):
    g = torch.Generator().manual_seed(1000 * Nq + Nk + D)
    r = lambda n: torch.randn((1, BH, n, D), generator=g)
    kv = (r(Nk) + 0.3 * torch.randn((1, BH, Nk, 1), generator=g)).to(dtype)
    q, do = r(Nq).to(dtype), r(Nq).to(dtype)
    dev = lambda t: t.to(DEV) if layout == "heads" else t.to(DEV).transpose(1, 2).contiguous().transpose(1, 2)   # tokens outside, heads inside
    return q, kv, do, dev(q), dev(kv), dev(do)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Nq", NQ)
def test_against_the_oracle(qfa, Nq, D):
    """dQ and dKV of three heads, for every number of keys; types and layouts by turns."""
    BH, sm = HEADS[D], 1.0 / math.sqrt(D)
    for i, Nk in enumerate(NK):
        dtype, sdtype = (torch.float16, torch.bfloat16)[(i + Nq) % 2], (torch.float16, torch.float32)[i // 2 % 2]
        q, kv, do, qd, kvd, dod = _case(BH, Nq, Nk, D, dtype, sdtype, ("heads", "tokens")[i // 3 % 2])
        assert skv_pass_takes(BH, Nq, Nk, D)
        qd.requires_grad_(True)
        kvd.requires_grad_(True)
        codes, scale, zp = qfa.asymmetric_quant_per_token(kvd.detach(), scale_dtype=sdtype)
        o = qfa.quant_flash_attn(qd, kvd, (codes, scale, zp), sm)
        grads = torch.autograd.grad(o, [qd, kvd], dod, retain_graph=True)
        again = torch.autograd.grad(o, [qd, kvd], dod)
        assert all(torch.equal(x, y) for x, y in zip(grads, again)), Nk
        pick = [0, BH // 2 + 1, BH - 1]
        q, do, codes, scale, zp, o, dq, dkv = (t.detach()[:, pick].cpu() for t in (q, do, codes, scale, zp, o, *grads))
        (dq_ref, dkv_ref), (nq, nkv) = oracle.legacy_bwd(q, codes, scale, zp, do, sm, o=o, spread=True)
        assert_close(f"dQ {Nk}", dq, dq_ref, scaled=True, spread=nq, cos_tol=COS_TOL if Nk > 1 else -1.0)   # one key: dQ is zero
        assert_close(f"dKV {Nk}", dkv, dkv_ref, scaled=True, spread=nkv)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Nq", [50, 100])
def test_scaled_beforehand_and_rows_that_are_not_finite(qfa, Nq, D):
    """dO in binary16 with a factor of its own beside it (the public call); an infinite query or dO row reaches dQ of its own
    query only, and other heads not at all."""
    BH, Nk, sm = HEADS[D], 150, 1.0 / math.sqrt(D)
    g = torch.Generator().manual_seed(D)
    kv, q, do = (torch.randn(s, generator=g).to(torch.float16).to(DEV) for s in ((1, BH, Nk, D), (1, BH, Nq, D), (1, BH, Nq, D)))
    codes, scale, zp = qfa.asymmetric_quant_per_token(kv)
    o, lse = qfa.attn_fwd_shared_kv(q, codes, scale, zp, sm)
    want = qfa.attn_bwd_shared_kv(q, codes, scale, zp, o, do, lse, sm)
    pick = [0, BH - 1]
    ref, spread = oracle.legacy_bwd(*(t[:, pick].cpu() for t in (q, codes, scale, zp, do)), sm, o=o[:, pick].cpu(), spread=True)
    for name, a, b, n in zip(("dQ", "dKV"), want, ref, spread):
        assert_close(name, a[:, pick].cpu(), b, scaled=True, spread=n)
    q2, do2 = q.clone(), do.clone()
    q2[:, 3, 40, 3] = float("inf")
    do2[:, 3, 7] = float("inf")
    o2, lse2 = qfa.attn_fwd_shared_kv(q2, codes, scale, zp, sm)
    got = qfa.attn_bwd_shared_kv(q2, codes, scale, zp, o2, do2, lse2, sm)
    keep = [i for i in range(Nq) if i not in (7, 40)]
    others = [h for h in range(BH) if h != 3]
    assert torch.isfinite(got[0][:, 3, keep]).all() and not torch.isfinite(got[1][:, 3]).all()
    for a, b in zip(got, want):
        assert torch.equal(a[:, others], b[:, others])


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Nq,Nk", [(40, 1025), (97, 1025), (40, 2049), (97, 2049)])
@pytest.mark.parametrize("dtype,sdtype", [(torch.float16, torch.float16), (torch.bfloat16, torch.float32)])
def test_a_large_scale_at_the_last_key(qfa, Nq, Nk, D, dtype, sdtype):
    """dO is scaled by what the largest key scale of the head leaves room for: the one that matters comes last, 2^14 times the others,
    where the scan for it starts another round of 1024 keys.  (Without it dP of that key is 5e8 and dS * scale 3e5: beyond binary16.)"""
    BH, sm = HEADS[D], 1.0 / math.sqrt(D)
    assert skv_pass_takes(BH, Nq, Nk, D)
    g = torch.Generator().manual_seed(Nq + Nk)
    kv = torch.randn((1, BH, Nk, D), generator=g) * 2.0 ** -6
    kv[:, :, -1] = 256.0 * (1.0 + 64.0 * kv[:, :, -1])
    q = (torch.randn((1, BH, Nq, D), generator=g) / 256.0).to(dtype)
    kv, do = kv.to(dtype), torch.full((1, BH, Nq, D), 2.0 ** -6, dtype=dtype)
    qd, kvd = q.to(DEV).requires_grad_(True), kv.to(DEV).requires_grad_(True)
    quant = qfa.asymmetric_quant_per_token(kvd.detach(), scale_dtype=sdtype)
    o = qfa.quant_flash_attn(qd, kvd, quant, sm)
    dq, dkv = torch.autograd.grad(o, [qd, kvd], do.to(DEV))
    assert torch.isfinite(dq).all() and torch.isfinite(dkv).all()
    pick = [0, BH - 1]
    q, do, codes, scale, zp, o, dq, dkv = (t.detach()[:, pick].cpu() for t in (q, do, *quant, o, dq, dkv))
    assert (scale[:, :, -1] > 1000 * scale[:, :, :-1].amax(2)).all()
    (dq_ref, dkv_ref), (nq, nkv) = oracle.legacy_bwd(q, codes, scale, zp, do, sm, o=o, spread=True)
    assert_close("dQ", dq, dq_ref, scaled=True, spread=nq)
    assert_close("dKV", dkv, dkv_ref, scaled=True, spread=nkv)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Nq", [50, 100])
def test_scales_of_zero_hide_nothing(qfa, Nq, D):
    """Keys whose scales are zero (a scale below binary16's range is stored as one) are keys: what is not finite in dO reaches dQ of its
    query through them, and a finite row's dQ is zero."""
    BH, Nk, sm = HEADS[D], 150, 1.0 / math.sqrt(D)
    g = torch.Generator().manual_seed(D)
    kv, q, do = (torch.randn(s, generator=g).to(torch.float16).to(DEV) for s in ((1, BH, Nk, D), (1, BH, Nq, D), (1, BH, Nq, D)))
    codes, scale, zp = qfa.asymmetric_quant_per_token(kv)
    scale[:, 3] = 0
    scale[:, 4, ::2] = 0
    do[:, 3:5, 7, 2] = float("inf")
    o, lse = qfa.attn_fwd_shared_kv(q, codes, scale, zp, sm)
    dq, dkv = qfa.attn_bwd_shared_kv(q, codes, scale, zp, o, do, lse, sm)
    rows = torch.isfinite(dq).all(-1)[0]
    want = torch.ones_like(rows)
    want[3:5, 7] = False
    assert torch.equal(rows, want)
    assert (dq[0, 3, :7] == 0).all() and (dq[0, 3, 8:] == 0).all()
    pick = [0, 5, BH - 1]
    ref, spread = oracle.legacy_bwd(*(t[:, pick].cpu() for t in (q, codes, scale, zp, do)), sm, o=o[:, pick].cpu(), spread=True)
    for name, a, b, n in zip(("dQ", "dKV"), (dq, dkv), ref, spread):
        assert_close(name, a[:, pick].cpu(), b, scaled=True, spread=n)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("which", ["codes", "dkv", "dq"])
def test_rows_far_apart(qfa, which, D):
    """Rows as far apart as the 31-bit offsets of the pass reach give the bits of dense ones; a step further the two kernels take the
    call, without scratch.  Their sums run in another order and the power of two that dO is scaled by is another one: the same
    products but for what binary16 loses (2^-10 of a value)."""
    BH, Nq, Nk = HEADS[D], 40, 1500
    L, g, sm = _lib.lib(), torch.Generator(device=DEV).manual_seed(D), 1.0 / math.sqrt(D)
    q, do = (torch.randn((1, BH, Nq, D), generator=g, device=DEV, dtype=torch.float16) for _ in range(2))
    kv = torch.randn((1, BH, Nk, D), generator=g, device=DEV, dtype=torch.float16)
    codes, scale, zp = qfa.asymmetric_quant_per_token(kv)
    o, lse = qfa.attn_fwd_shared_kv(q, codes, scale, zp, sm)

    def apart(t, stride):   # the same tensor (or room for it) with tokens `stride` elements apart, the heads of a token side by side
        x = torch.empty((t.size(2) - 1) * stride + BH * D, dtype=t.dtype, device=DEV).as_strided(t.shape, (BH * D, D, stride, 1))
        return x.copy_(t)

    def run(codes, dq, dkv):
        st = lambda t: t.stride()[:3]
        rc = L.qfa_attn_bwd_shared_kv_direct(q.data_ptr(), codes.data_ptr(), scale.data_ptr(), 1, zp.data_ptr(), o.data_ptr(), do.data_ptr(),
                                             lse.data_ptr(), dq.data_ptr(), dkv.data_ptr(), 1, 1, 1, 1, BH, Nq, Nk, D, *st(q), *st(codes),
                                             *st(o), *st(do), *st(dq), *st(dkv), sm, None, 0, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, L.qfa_last_error()
        return dq, dkv
    want = run(codes, torch.zeros_like(q), torch.zeros_like(kv))
    rows = Nk + 512
    past = {"codes": -(-(1 << 31) // rows), "dkv": -(-(1 << 30) // rows), "dq": 1 << 23}[which]   # the first stride that does not fit
    past = -(-past // 16) * 16
    for stride in (past - 16, past):
        args = [codes, torch.zeros_like(q), torch.zeros_like(kv)]
        i = ["codes", "dq", "dkv"].index(which)
        args[i] = apart(args[i], stride)
        got = run(*args)
        assert all(torch.equal(a, b) for a, b in zip(got, want)) == (stride < past)
        for a, b in zip(got, want):
            assert (a.double() - b.double()).norm() <= 2.0 ** -9 * b.double().norm()
