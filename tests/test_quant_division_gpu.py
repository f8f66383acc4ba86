"""The quantizer's division by a token's scale, as its kernels compute it, against the IEEE division: every pair of an 11-bit
significand (16-bit tensors, one residual correction) with a scale's, and pairs with 24-bit significands (two)."""
import ctypes
import os
import subprocess

import pytest
import torch

from quant_flash_attn_amd import build

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native")
LIB = os.path.join(HERE, "libquant_division.so")


def build_library():
    cmd = [build._hipcc(), *build.COMMON, "-ffp-contract=off", "-fno-fast-math", "-shared", "-x", "hip",
           os.path.join(HERE, "quant_division.hip"), "-o", LIB]
    subprocess.run(cmd, check=True, capture_output=True)


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(LIB):
        build_library()
    handle = ctypes.CDLL(LIB)
    handle.compare_quotients.argtypes = [ctypes.c_int, ctypes.c_uint, ctypes.c_void_p, ctypes.c_void_p]
    return handle


def _wrong(lib, short, offset):
    count = torch.zeros(1, dtype=torch.int64, device="cuda:0")
    assert lib.compare_quotients(short, offset, count.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    return int(count.cpu())


@pytest.mark.gpu
def test_one_correction_for_16_bit_elements(lib):
    assert _wrong(lib, 1, 0) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("offset", [0, 1, 4095, 4097, 8191])
def test_two_corrections_for_fp32_elements(lib, offset):
    assert _wrong(lib, 0, offset) == 0
