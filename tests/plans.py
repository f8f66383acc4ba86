"""What the library's planning functions (C++, pure functions of the sizes) decide, so that a test can say which kernels a case is
to reach (not collected by pytest)."""
import ctypes

from quant_flash_attn_amd import _lib

_L, _I = ctypes.c_int64, ctypes.c_int


class BwdPlan(ctypes.Structure):
    _fields_ = [(n, _I) for n in ("blocks_dkv", "splits_dkv", "queries_per_split", "blocks_dq", "splits_dq", "keys_per_split",
                                  "sum_between")] + [("part_bytes", _L)]


class SkvTilePlan(ctypes.Structure):
    _fields_ = [(n, _I) for n in ("waves", "splits", "tiles")]   # waves side by side; 0: the 16-query kernel


class SkvFwdPlan(ctypes.Structure):
    _fields_ = [("tile", SkvTilePlan), ("splits", _I), ("tiles_per_split", _I), ("part_bytes", _L)]


def _plan(name, result, args):
    f = getattr(_lib.lib(), name)
    f.restype, f.argtypes = result, args
    return f


def fwd_o_once(BH, Nq, Nk, D, o, strides):
    """whether the forward's O at address `o` is written past the caches; strides of its [B, H, N] in elements"""
    return _plan("_ZN3qfa10fwd_o_onceEllliPKvlll", ctypes.c_bool, [_L, _L, _L, _I, ctypes.c_void_p, _L, _L, _L])(BH, Nq, Nk, D, o, *strides)


def bwd_plan(BH, Nq, Nk, D, causal, may_split=1):
    return _plan("_ZN3qfa8bwd_planEllliii", BwdPlan, [_L, _L, _L, _I, _I, _I])(BH, Nq, Nk, D, int(causal), may_split)


def bwd_plan_within(BH, Nq, Nk, D, causal, room):
    """what a call with `room` bytes for parts launches"""
    return _plan("_ZN3qfa15bwd_plan_withinEllliil", BwdPlan, [_L, _L, _L, _I, _I, _L])(BH, Nq, Nk, D, int(causal), room)


def skv_tile_fwd_plan(BH, Nq, Nk, D):
    return _plan("_ZN3qfa12skv_fwd_planEllli", SkvFwdPlan, [_L, _L, _L, _I])(BH, Nq, Nk, D).tile


def skv_tile_dq_plan(BH, Nq, Nk, D):
    return _plan("_ZN3qfa16skv_tile_dq_planEllli", SkvTilePlan, [_L, _L, _L, _I])(BH, Nq, Nk, D)


def skv_pass_takes(BH, Nq, Nk, D):
    return _plan("_ZN3qfa14skv_pass_takesEllli", ctypes.c_bool, [_L, _L, _L, _I])(BH, Nq, Nk, D)


def skv_pass_takes_unsplit(BH, Nq, Nk, D):
    return _plan("_ZN3qfa22skv_pass_takes_unsplitEllli", ctypes.c_bool, [_L, _L, _L, _I])(BH, Nq, Nk, D)
