"""Whether the forward writes O past the caches: beyond the last-level cache, and in whole lines."""
import os

import pytest

from plans import fwd_o_once
from quant_flash_attn_amd import build

AT = 1 << 30   # (an address; nothing is read)


@pytest.mark.parametrize("D", [128, 256])
def test_whole_lines_beyond_the_last_level_cache(qfa, D):
    H, N = 31 * 58, 231
    assert H * 2 * N * D * 3 > 256 << 20
    head_major, token_major, padded = (H * N * D, N * D, D), (H * N * D, D, H * D), (H * N * (D + 8), N * (D + 8), D + 8)
    assert fwd_o_once(H, N, N, D, AT, head_major) and fwd_o_once(H, N, N, D, AT, token_major)
    assert fwd_o_once(H, N, N, D, AT + 16, head_major)            # (in one piece: two heads share a line at most)
    assert not fwd_o_once(H, N, N, D, AT + 16, token_major)       # 1.025 to 1.05 times as long with the hint
    assert not fwd_o_once(H, N, N, D, AT, padded)                 # 1.004 to 1.05
    assert not fwd_o_once(H // 8, N, N, D, AT, head_major)
    assert not fwd_o_once(4 * H, N, N, 64, AT, (4 * H * N * 64, N * 64, 64))


def test_the_compiler_kept_both_stores(qfa):
    """(it makes one of two stores that differ in the hint only, without it)"""
    asm = build.assembly_path("qfa_fwd_wide.hip")
    if not os.path.exists(asm):
        pytest.skip("the library's assembly is not there: it stays in the build folder of the machine that built it")
    stores = [line for line in open(asm) if "global_store_dwordx4" in line]
    assert 0 < sum(line.split()[-1] == "nt" for line in stores) < len(stores)
