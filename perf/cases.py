"""The work a user of this framework has it do, as timed cases through the public entry points.

Four families, each over the range of sizes it is used at:

  qkv       quant_flash_attn_qkv: training (forward + backward) and prefill (forward) on 16-bit or fp32 q, k, v
  cache     quant_flash_attn_quantized_kv: queries at the end of an INT8 K / V cache -- one token (decode), a few, or
            a chunk of a prompt (prefill in pieces); the mask is aligned to the last key
  shared    quant_flash_attn: the reference's own operator, one quantized tensor as K and V (training and decode)
  quantize  asymmetric_quant_per_token: a K or V tensor on its way into the cache

A case's fields: kind, B, H, Nq, Nk, D, dtype, and where they apply causal, grad (forward + backward) and dist.
"""
import math

import torch

import quant_flash_attn_amd as qfa

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# Bounds of a drawn case: what the largest listed ones cost.
_MAX_FLOPS = 7.7e12
_MAX_BYTES = 8.0e9


def listed():
    return [
        # The smallest call: one short sequence of a small fp32 model, trained.  Latency, launches and host time.
        dict(name="small_fp32_train", kind="qkv", B=1, H=4, Nq=256, Nk=256, D=64, dtype="fp32", causal=False, grad=True,
             dist="normal"),
        # Prefill of four 4096-token sequences with 32 heads of 128: the configuration of the headline metric.
        dict(name="prefill_d128", kind="qkv", B=4, H=32, Nq=4096, Nk=4096, D=128, dtype="bf16", causal=True, grad=False,
             dist="offset"),
        # The same configuration trained (the metric's second half).
        dict(name="train_d128", kind="qkv", B=4, H=32, Nq=4096, Nk=4096, D=128, dtype="bf16", causal=True, grad=True,
             dist="offset"),
        # One long sequence, no mask, keys with outlier channels.
        dict(name="long_context_train", kind="qkv", B=1, H=16, Nq=16384, Nk=16384, D=128, dtype="bf16", causal=False,
             grad=True, dist="outlier"),
        # A batch of medium sequences with small heads.
        dict(name="train_d64", kind="qkv", B=16, H=16, Nq=2048, Nk=2048, D=64, dtype="bf16", causal=True, grad=True,
             dist="uniform"),
        # The widest heads.
        dict(name="train_d256", kind="qkv", B=4, H=16, Nq=4096, Nk=4096, D=256, dtype="bf16", causal=True, grad=True,
             dist="offset"),
        # A piece of a prompt appended to a cache of several thousand tokens; no length is a multiple of a tile.
        dict(name="cache_chunk", kind="cache", B=2, H=32, Nq=333, Nk=7001, D=128, dtype="bf16", causal=True, grad=False,
             dist="offset"),
        # One decoding step of a batch of eight sequences with an INT8 cache.
        dict(name="cache_decode", kind="cache", B=8, H=32, Nq=1, Nk=8192, D=128, dtype="bf16", causal=True, grad=False,
             dist="offset"),
        # The reference's benchmark shape (compute_flops.py:96): very many short query blocks, forward and backward.
        dict(name="shared_bench", kind="shared", B=512, H=16, Nq=16, Nk=3000, D=128, dtype="fp16", causal=False, grad=True,
             dist="normal"),
        # The reference's accuracy-test shape (test_accuracy.py:44): odd sizes everywhere.
        dict(name="shared_ragged", kind="shared", B=99, H=53, Nq=97, Nk=689, D=128, dtype="fp16", causal=False, grad=True,
             dist="normal"),
        # One decoding step of one sequence with a long shared-KV cache.
        dict(name="shared_decode", kind="shared", B=1, H=32, Nq=1, Nk=32768, D=128, dtype="bf16", causal=False, grad=False,
             dist="normal"),
        # The reference's quantizer benchmark (asymmetric_quant.py:196-207).
        dict(name="quantize", kind="quantize", B=8, H=32, Nq=4096, Nk=4096, D=128, dtype="fp16", causal=False, grad=False,
             dist="normal"),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["qkv", "qkv", "qkv", "cache", "cache", "shared", "shared", "quantize"])
    c = dict(kind=kind, B=_log(rng, 1, 32), H=_log(rng, 1, 64), D=rng.choice([64, 128, 128, 256]),
             dtype=rng.choice(["bf16", "bf16", "fp16"]), causal=False, grad=False, dist=rng.choice(["normal", "offset", "outlier", "uniform"]))
    if kind == "qkv":
        c["Nk"] = c["Nq"] = _log(rng, 64, 16384)
        if rng.random() < 0.2:                      # fewer queries than keys
            c["Nq"] = _log(rng, max(1, c["Nk"] // 16), c["Nk"])
        c["causal"], c["grad"] = rng.random() < 0.6, rng.random() < 0.6
        if rng.random() < 0.1:
            c["dtype"] = "fp32"
    elif kind == "cache":
        c["Nk"] = _log(rng, 256, 32768)
        c["Nq"] = rng.choice([1, 1, _log(rng, 2, 16), _log(rng, 16, 2048)])
        c["Nq"] = min(c["Nq"], c["Nk"])
        c["causal"] = True
    elif kind == "shared":
        c["grad"] = rng.random() < 0.6
        c["B"] = _log(rng, 1, 512)
        c["Nk"] = _log(rng, 256, 32768)
        c["Nq"] = _log(rng, 1, 512)
    else:
        c["Nk"] = c["Nq"] = _log(rng, 64, 16384)
        c["dtype"] = rng.choice(["bf16", "fp16", "fp32"])
        c["D"] = rng.choice([64, 96, 128, 256])
    while True:                                     # no more work than the largest listed case
        w = work(c)
        if w["flops"] <= _MAX_FLOPS and w["bytes"] <= _MAX_BYTES:
            return c
        key = "B" if c["B"] > 1 else "H" if c["H"] > 1 else "Nk"
        c[key] = max(1, int(c[key] / 1.4))
        if key == "Nk":
            c["Nq"] = min(c["Nq"], c["Nk"])


def _values(g, dist, shape, dtype):
    """N(0,1) activations; 'offset': a mean per token (zero points away from zero); 'outlier': one channel in a hundred
    five times as large; 'uniform': U(-1, 2)."""
    if dist == "uniform":
        return (torch.rand(shape, generator=g, device="cuda", dtype=torch.float32) * 3.0 - 1.0).to(dtype)
    x = torch.randn(shape, generator=g, device="cuda", dtype=dtype)
    if dist == "offset":
        x += 0.3 * torch.randn(shape[:3] + (1,), generator=g, device="cuda", dtype=dtype)
    elif dist == "outlier":
        x[..., :max(1, math.ceil(0.01 * shape[3]))] *= 5.0
    return x


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    B, H, Nq, Nk, D = (case[k] for k in ("B", "H", "Nq", "Nk", "D"))
    dt, dist, grad = _DTYPES[case["dtype"]], case["dist"], case["grad"]
    # outlier channels are the keys' (scores stay of the size a trained model has); values are plain or have a mean
    qdist, vdist = ("normal" if dist == "outlier" else dist), (dist if dist == "offset" else "normal")
    s = dict(kind=case["kind"], causal=case["causal"], grad=grad, sm=1.0 / math.sqrt(D))
    if case["kind"] == "quantize":
        s["x"] = _values(g, dist, (B, H, Nk, D), dt)
        return s
    s["q"] = _values(g, qdist, (B, H, Nq, D), dt)
    if case["kind"] == "qkv":
        s["k"] = _values(g, dist, (B, H, Nk, D), dt)
        s["v"] = _values(g, vdist, (B, H, Nk, D), dt)
        leaves = ("q", "k", "v")
    elif case["kind"] == "cache":
        # the cache holds codes only; the 16-bit placeholders of the entry point are empty
        s["k_quant"] = qfa.asymmetric_quant_per_token(_values(g, dist, (B, H, Nk, D), dt))
        s["v_quant"] = qfa.asymmetric_quant_per_token(_values(g, vdist, (B, H, Nk, D), dt))
        s["none"] = torch.empty(0, dtype=dt, device="cuda")
        leaves = ()
    else:
        kv = _values(g, dist, (B, H, Nk, D), dt)
        s["kv_quant"] = qfa.asymmetric_quant_per_token(kv)
        s["kv"] = kv            # the leaf that receives the gradient
        leaves = ("q", "kv")
    if grad:
        s["do"] = torch.randn((B, H, Nq, D), generator=g, device="cuda", dtype=dt)
        for name in leaves:
            s[name].requires_grad_(True)
        s["leaves"] = leaves
    return s


def _forward(s):
    if s["kind"] == "qkv":
        return qfa.quant_flash_attn_qkv(s["q"], s["k"], s["v"], s["causal"], s["sm"])
    if s["kind"] == "cache":
        return qfa.quant_flash_attn_quantized_kv(s["q"], s["none"], s["none"], s["k_quant"], s["v_quant"], s["causal"], s["sm"])
    return qfa.quant_flash_attn(s["q"], s["kv"], s["kv_quant"], s["sm"])


def run(state):
    if state["kind"] == "quantize":
        return qfa.asymmetric_quant_per_token(state["x"])
    if not state["grad"]:
        with torch.no_grad():
            return _forward(state)
    o = _forward(state)
    return (o.detach(),) + torch.autograd.grad(o, [state[n] for n in state["leaves"]], state["do"])


def work(case):
    B, H, Nq, Nk, D = (case[k] for k in ("B", "H", "Nq", "Nk", "D"))
    es = 4 if case["dtype"] == "fp32" else 2
    row = H * D * B
    if case["kind"] == "quantize":
        # codes, fp16 scale, zero point; per element a quotient, an addition and a rounding
        return {"bytes": row * Nk * (es + 1) + B * H * Nk * 3, "flops": 3.0 * row * Nk}
    pairs = Nq * Nk - (Nq * (Nq - 1) // 2 if case["causal"] else 0)   # (query, key) pairs the mask leaves
    flops = 4.0 * row * pairs * (3.5 if case["grad"] else 1.0)       # backward 2.5 x forward (compute_flops.py:103-104)
    code = row * Nk + B * H * Nk * 3                                  # a quantized tensor: codes, fp16 scale, zero point
    qo = 2 * row * Nq * es                                            # q and o
    if case["kind"] == "qkv":
        bytes_ = qo + 2 * row * Nk * es
        if case["grad"]:
            bytes_ *= 2                                               # dO, dQ, dK, dV
    elif case["kind"] == "cache":
        bytes_ = qo + 2 * code
    else:
        bytes_ = qo + code
        if case["grad"]:
            bytes_ += qo + row * Nk * es                              # dO, dQ; dKV
    return {"bytes": float(bytes_), "flops": flops}


def tolerance(case):
    if case["kind"] == "quantize":
        return "exact"
    # probabilities and score gradients pass through the 16-bit type (fp32 tensors through bf16); the shared-KV
    # backward computes in binary16 whatever the tensors' type
    return {"rel": 3e-3} if case["dtype"] == "fp16" else {"rel": 1e-2}
