"""Builds quant_flash_attn_amd/libqfa.so from csrc/ with hipcc for gfx950, and the module of its host path.

    python -m quant_flash_attn_amd.build          # compile every translation unit, then link

libqfa.so holds the kernels behind the C ABI; _qfa_host.so (csrc/qfa_torch.cpp, host code only, against torch's headers)
is what the Python entry points call.  Both are built in-tree so that a source snapshot carries it along; nothing is
JIT-compiled at import time.  Compilation needs no GPU (hipcc cross-compiles).
"""
from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
import tempfile
from concurrent.futures import ThreadPoolExecutor

from . import acc_check

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libqfa.so")
HOST_MODULE = os.path.join(HERE, "_qfa_host.so")
OBJ_DIR = os.path.join(HERE, "build")

# -packed-fp32-ops: keep hipcc from forming v_pk_*_f32 out of scalar float code.
COMMON = ["--offload-arch=gfx950", "-O3", "-fPIC", "-std=c++17", "-Wall", "-Wno-unused-function",
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
# whatever quantizes must evaluate its expressions as single IEEE operations (bit-exact codes)
PER_FILE = {f: ["-ffp-contract=off", "-fno-fast-math"] for f in ("qfa_quant.hip", "qfa_cache.hip")}
# accumulators in AccVGPRs by hand (see qfa_acc.h): other MFMA results in vector registers, and the assembly is checked
_BWD_PAIR = tuple(f"qfa_bwd_pair_{x}.hip" for x in ("128_bf16", "128_f16", "256_bf16", "256_f16", "64_bf16", "64_f16"))
BY_HAND = ("qfa_fwd_wide.hip", *_BWD_PAIR, "qfa_skv_pass.hip")
# MFMA results in vector registers: head_dim 256 with four waves side by side then spills none instead of 5 (dQ) and 1 instead of 4 (forward);
# elsewhere only the forward of 64 with four waves does, 4 registers, with and without (dKV: no difference in registers)
PER_FILE["qfa_skv_tile.hip"] = PER_FILE["qfa_skv_dkv.hip"] = PER_FILE["qfa_skv_pass64.hip"] = ["-mllvm", "-amdgpu-mfma-vgpr-form"]
for _f in BY_HAND:
    PER_FILE[_f] = ["-mllvm", "-amdgpu-mfma-vgpr-form"]
SOURCES = ["qfa_api.cpp", "qfa_quant.hip", "qfa_fwd.hip", "qfa_fwd_wide.hip", "qfa_split_plan.cpp", "qfa_bwd.hip", *_BWD_PAIR, "qfa_skv_plan.cpp", "qfa_skv.hip", "qfa_skv_tile.hip", "qfa_skv_dkv.hip", "qfa_skv_pass.hip", "qfa_skv_pass64.hip", "qfa_skv_bwd.hip", "qfa_skv_bwd_long.hip",
           "qfa_cache.hip"]


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.isabs(cand) and os.path.exists(cand) or not os.path.isabs(cand)):
            return cand
    raise RuntimeError("hipcc not found")


def _compile(src: str, extra=()) -> str:
    obj = os.path.join(OBJ_DIR, os.path.splitext(src)[0] + ".o")
    cmd = [_hipcc(), *COMMON, *PER_FILE.get(src, []), *extra, "-x", "hip", "-c", os.path.join(CSRC, src), "-o", obj]
    if src in BY_HAND:
        return _compile_checked(src, cmd, obj)
    _run(src, cmd)
    return obj


def assembly_path(src: str) -> str:
    """The device assembly that the build keeps of a file in BY_HAND."""
    return os.path.join(OBJ_DIR, os.path.splitext(src)[0] + ".s")


def _compile_checked(src: str, cmd, obj: str) -> str:
    with tempfile.TemporaryDirectory(dir=OBJ_DIR) as tmp:
        made = os.path.join(tmp, os.path.basename(obj))
        _run(src, [*cmd[:-1], made, "--save-temps=obj"])
        asm, = (f for f in os.listdir(tmp) if f.endswith("gfx950.s"))
        os.replace(os.path.join(tmp, asm), assembly_path(src))
        found = acc_check.check(assembly_path(src))
        if found:
            raise RuntimeError(f"{src}: the compiler's output breaks the rules of qfa_acc.h:\n" + "\n".join(found))
        os.replace(made, obj)
    return obj


def _run(src: str, cmd) -> None:
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{res.stdout}\n{res.stderr}")
    # hipcc's host pass warns that it does not know the packed-fp32 feature: harmless, not shown
    noise = ("packed-fp32-ops", "is not a recognized feature")
    for line in res.stderr.splitlines():
        if line.strip() and not any(n in line for n in noise):
            print(line, file=sys.stderr)


def _compile_host_module() -> str:
    import torch
    root = os.path.dirname(torch.__file__)
    inc = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
           sysconfig.get_paths()["include"], os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include")]
    tmp = HOST_MODULE + ".tmp"
    cmd = ["g++", "-O2", "-fPIC", "-shared", "-std=c++17", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           "-DTORCH_API_INCLUDE_EXTENSION_H", "-DTORCH_EXTENSION_NAME=_qfa_host",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *(x for i in inc for x in ("-isystem", i)),
           os.path.join(CSRC, "qfa_torch.cpp"), "-o", tmp, "-L" + os.path.join(root, "lib"), "-lc10", "-lc10_hip",
           "-ltorch_cpu", "-ltorch", "-ltorch_python"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed for qfa_torch.cpp:\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, HOST_MODULE)
    return HOST_MODULE


def build_library(extra_flags=(), jobs: int = 4) -> str:
    os.makedirs(OBJ_DIR, exist_ok=True)
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        host = pool.submit(_compile_host_module)
        objs = list(pool.map(lambda s: _compile(s, extra_flags), SOURCES))
    tmp = LIB + ".tmp"
    res = subprocess.run([_hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *objs],
                         capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stdout}\n{res.stderr}")
    host.result()
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build_library())
