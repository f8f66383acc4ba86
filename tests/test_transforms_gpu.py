"""The entry points under torch's function transforms: a traced call runs the operator again (with its gradient), a tensor
that carries a forward-mode tangent is refused, since the operators have no forward-mode derivative."""
import math

import pytest
import torch

from quant_flash_attn_amd.synthetic import make_inputs

DEV = "cuda:0"
SM = 1.0 / math.sqrt(64)


def _inputs(qfa, Nq, seed, device=DEV):
    q, k, v, _ = (t.to(device) for t in make_inputs("offset", 1, 2, 96, 64, seed=seed, dtype=torch.float16))
    return q[:, :, :Nq].contiguous(), k, v


def _calls(qfa):
    """name -> (function of the tensors, longest query block in use): every route behind the entry points."""
    def quantized(q, k, v, *codes):
        return qfa.quant_flash_attn_quantized_kv(q, k, v, codes[:3], codes[3:], True, SM)

    def shared(q, kv, *codes):
        return qfa.quant_flash_attn(q, kv, codes, SM)

    return {"qkv": lambda q, k, v: qfa.quant_flash_attn_qkv(q, k, v, True, SM), "cache": quantized, "shared": shared}


def _args(qfa, name, Nq, seed):
    q, k, v = _inputs(qfa, Nq, seed)
    if name == "qkv":
        return q, k, v
    kq = qfa.asymmetric_quant_per_token(k)
    if name == "shared":
        return (q, k) + tuple(kq)
    return (q, k, v) + tuple(kq) + tuple(qfa.asymmetric_quant_per_token(v))


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["qkv", "cache", "shared"])
@pytest.mark.parametrize("grad", [False, True])
def test_a_traced_call_computes(qfa, name, grad):
    call = _calls(qfa)[name]
    args = _args(qfa, name, 48, seed=1)
    leaves = 2 if name == "shared" else 3
    if grad:
        for t in args[:leaves]:
            t.requires_grad_(True)
    traced = torch.jit.trace(call, args, check_trace=False)
    for seed in (1, 2):
        fresh = _args(qfa, name, 48, seed)
        if grad:
            for t in fresh[:leaves]:
                t.requires_grad_(True)
        got, want = traced(*fresh), call(*fresh)
        assert torch.equal(got, want)
        if grad:
            do = torch.randn_like(want)
            for a, b in zip(torch.autograd.grad(got, fresh[:leaves], do), torch.autograd.grad(want, fresh[:leaves], do)):
                assert torch.equal(a, b)


def _refused(call, args, which):
    import torch.autograd.forward_ad as fwAD
    with fwAD.dual_level():
        dual = list(args)
        dual[which] = fwAD.make_dual(args[which], torch.ones_like(args[which]))
        with pytest.raises(NotImplementedError):
            call(*dual)
        with torch.no_grad(), pytest.raises(NotImplementedError):
            call(*dual)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["qkv", "cache", "shared"])
def test_forward_mode_is_refused(qfa, name):
    args = _args(qfa, name, 48, seed=1)
    for which in range(2 if name == "shared" else 3):
        _refused(_calls(qfa)[name], args, which)


def test_forward_mode_is_refused_whatever_the_device(qfa):
    q = torch.zeros(1, 1, 4, 64, dtype=torch.float16)
    codes = (torch.zeros(1, 1, 4, 64, dtype=torch.int8), torch.ones(1, 1, 4, 1), torch.zeros(1, 1, 4, 1, dtype=torch.int8))
    for which in range(3):
        _refused(_calls(qfa)["qkv"], (q, q.clone(), q.clone()), which)
        _refused(_calls(qfa)["cache"], (q, q.clone(), q.clone()) + codes + codes, which)
    for which in range(2):
        _refused(_calls(qfa)["shared"], (q, q.clone()) + codes, which)
