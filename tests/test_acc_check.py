"""The build's check of hand-kept accumulators: it finds each fault in a few lines of assembly that hold it, and nothing in the
assembly of the library as it was built."""
import os

import pytest

from quant_flash_attn_amd import acc_check, build

MFMA = "v_mfma_f32_32x32x16_bf16 a[0:15], v[0:3], v[4:7], a[0:15]"
READ = "v_accvgpr_read_b32 v9, a3"


def _kernel(tmp_path, *lines, scratch=0):
    """Lines that begin with '!' come from inline assembly."""
    out = ["_Zkernel:"]
    for line in lines:
        out += ["\t;;#ASMSTART", "\t" + line[1:], "\t;;#ASMEND"] if line.startswith("!") else [line if line.endswith(":") else "\t" + line]
    out += ["\ts_endpgm", f"\t\t.amdhsa_private_segment_fixed_size {scratch}"]
    path = tmp_path / "k.s"
    path.write_text("\n".join(out) + "\n")
    return acc_check.check(str(path))


@pytest.mark.parametrize("between,ok", [([], False), (["s_mov_b32 s0, 0"], False), (["s_nop 0"], False), (["s_nop 1"], True),
                                        (["v_mov_b32_e32 v20, v21", "s_mov_b32 s0, 0"], True), ([".LBB0_1:"], False)])
@pytest.mark.parametrize("write", ["v_cvt_pk_bf16_f32 v7, v8, v9", "v_mov_b64_e32 v[2:3], v[8:9]", "v_permlane32_swap_b32_e32 v30, v4"])
def test_operand_written_just_before_its_mfma(tmp_path, write, between, ok):
    assert (not _kernel(tmp_path, write, *between, "!" + MFMA)) == ok


def test_operand_written_at_the_end_of_a_loop(tmp_path):
    loop = [".LBB0_1:", "!" + MFMA, "v_cvt_pk_bf16_f32 v7, v8, v9"]
    assert _kernel(tmp_path, *loop, "s_cbranch_scc1 .LBB0_1")
    assert not _kernel(tmp_path, *loop, "s_nop 0", "s_cbranch_scc1 .LBB0_1")
    assert not _kernel(tmp_path, *loop, "s_branch .LBB0_2", ".LBB0_2:")


def test_operands_that_loads_write_are_not_the_rule_s(tmp_path):
    assert not _kernel(tmp_path, "ds_read_b128 v[0:3], v50", "s_waitcnt lgkmcnt(0)", "!" + MFMA)
    assert not _kernel(tmp_path, "ds_write_b128 v60, v[0:3]", "!" + MFMA)
    assert _kernel(tmp_path, "v_mfma_f32_32x32x16_bf16 v[0:15], v[20:23], v[24:27], 0", "s_nop 7", "!" + MFMA)


@pytest.mark.parametrize("wait,ok", [([], False), (["!s_nop 15"], False), (["!s_nop 15", "!s_nop 15"], True)])
@pytest.mark.parametrize("use", [READ, "v_accvgpr_write_b32 a15, v9"])
def test_accumulator_used_before_its_mfma_is_done(tmp_path, use, wait, ok):
    assert (not _kernel(tmp_path, "!" + MFMA, *wait, "!" + use)) == ok


@pytest.mark.parametrize("line,ok", [("v_accvgpr_write_b32 a15, v9", False), ("v_accvgpr_read_b32 v9, a0", False),
                                     ("global_load_dwordx4 a[12:15], v[8:9], off", False), ("v_mov_b32_e32 v9, v8", True),
                                     ("v_accvgpr_write_b32 a16, v9", True), ("ds_write_b128 v9, a[16:19]", True)])
@pytest.mark.parametrize("place", [0, 2])
def test_the_compiler_in_an_accumulator(tmp_path, line, ok, place):
    lines = ["!" + MFMA, "s_nop 15", "s_nop 15", "!" + MFMA]
    lines.insert(place, line)
    assert (not _kernel(tmp_path, *lines)) == ok


def test_scratch(tmp_path):
    assert _kernel(tmp_path, "!" + MFMA, scratch=16)
    assert not _kernel(tmp_path, "v_mov_b32_e32 v9, v8", scratch=16)   # no accumulators by hand: not its business


@pytest.mark.parametrize("src", build.BY_HAND)
def test_the_library_as_built(src):
    asm = build.assembly_path(src)
    if not os.path.exists(asm):
        pytest.skip("the library's assembly is not there: it stays in the build folder of the machine that built it")
    assert acc_check.check(asm) == []
    text = open(asm).read()
    assert text.count("_kernel") > 0 and "ASMSTART" in text


def test_a_register_named_in_brackets(tmp_path):
    assert _kernel(tmp_path, "!" + MFMA, "!v_accvgpr_read_b32 v9, a[3]")
    assert not _kernel(tmp_path, "!" + MFMA, "!v_accvgpr_read_b32 v9, a[16]")


def test_two_loops_of_which_a_workgroup_runs_one(tmp_path):
    """The second one's accumulators are the compiler's in the first, also where a path leads on from it, as long as they begin anew."""
    other = "v_mfma_f32_32x32x16_bf16 a[16:31], v[0:3], v[4:7], a[16:31]"
    zero = [f"!v_accvgpr_write_b32 a[{r}], 0" for r in range(16, 32)]
    first = ["s_cbranch_scc1 .LBB0_2", "v_accvgpr_write_b32 a16, v9", "s_nop 1", "!" + MFMA, "v_accvgpr_read_b32 v9, a16"]
    assert not _kernel(tmp_path, *first, ".LBB0_2:", *zero, "s_nop 1", "!" + other)
    assert _kernel(tmp_path, *first, ".LBB0_2:", *zero[1:], "s_nop 1", "!" + other)
    assert _kernel(tmp_path, *first[:-1], "!" + zero[0][1:], first[-1])   # the compiler's value is gone
