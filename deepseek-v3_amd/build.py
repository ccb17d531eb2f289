"""Builds libdsv3fp8.so (HIP kernels + C ABI) for gfx950 with hipcc and libdsv3torch.so (the native part of the torch
operators, on top of it) with the host compiler, in-tree.

    python deepseek-v3_amd/build.py            # build into deepseek-v3_amd/lib/
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

HERE = Path(__file__).resolve().parent
CSRC = HERE / "csrc"
LIB_DIR = HERE / "lib"
LIB_PATH = LIB_DIR / "libdsv3fp8.so"
TORCH_SRC = CSRC / "torch_ops.cpp"
TORCH_LIB_PATH = LIB_DIR / "libdsv3torch.so"

ARCH = "gfx950"
# -packed-fp32-ops off: the compiler must not form v_pk_{add,mul,fma}_f32 from scalar float code.
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument", "-Wno-unknown-warning-option",
    "-fno-fast-math", "-ffp-contract=off",
]


# The decode kernels of these files must not use scratch memory, for two reasons.  Some of them issue their global
# loads and count the outstanding ones by hand (inline asm global_load + s_waitcnt vmcnt(n)): the register named by
# such a load is not valid until the wait, so a spill or a copy of it in between would read the register before the
# data has landed.  And a kernel that uses scratch at all costs a launch about 3 us more on this hardware (measured:
# linear() at one row 7.4 -> 10.4 us when a rewrite of the in-kernel quantiser spilled nine registers) -- as much as
# the whole quantisation such a launch is meant to save.  The build fails if a kernel of these files reports scratch
# or spills; exceptions are listed with their reasons.
# The attention kernels keep their sums in registers for a whole loop and have none to spare (mla_decode_kernel: 32 x 512
# sums in the 256 accumulation registers; an ordinary rescale of them spilled 300): a spill there is a copy per tile.
NO_SPILL_SOURCES = {"fp8_gemm_skinny.hip", "fp8_gemm_stream.hip", "fp8_gemm_mid.hip", "mla_decode.hip", "mla_prefill.hip"}
SGPR_SPILLS_ALLOWED = {
    # Scalars kept in lanes of a vector register are no scratch memory and cost nothing outside the tile loop: the limit for them.  (This build
    # reports none.)  The kernel takes all 256 vector registers, so a spilled one of these would be a copy per tile: refused.
    "mla_attend_kernel": 2,
}
SCRATCH_ALLOWED = {
    # the quantising variant with four strips per wavefront (a plan for very wide weights at one or two rows that none
    # of the 671B projections takes): compiler-counted waits, 20 bytes per lane
    "skinny_kernelILi1ELi4ELi2ELb1ELb0E": 24,
}


def check_no_spills(name: str, remarks: str) -> None:
    import re
    kernel = None
    for line in remarks.splitlines():
        m = re.search(r"Function Name: (\S+)", line)
        if m:
            kernel = m.group(1)
            continue
        m = re.search(r"(VGPRs Spill|SGPRs Spill|ScratchSize \[bytes/lane\]): (\d+)", line)
        if not (m and kernel and "_kernel" in kernel):
            continue
        exceptions = {**SCRATCH_ALLOWED, **(SGPR_SPILLS_ALLOWED if m.group(1) == "SGPRs Spill" else {})}
        allowed = max([v for k, v in exceptions.items() if k in kernel], default=0)
        if int(m.group(2)) > allowed:
            raise RuntimeError(f"{name}: {kernel} reports {m.group(1)} = {m.group(2)} (allowed: {allowed}); these "
                               f"kernels must not spill (lower the kernel's register use or its occupancy target)")


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found: cannot build libdsv3fp8.so")
    return exe


def sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip"))


def build_library(verbose: bool = True) -> Path:
    hipcc = _hipcc()
    obj_dir = HERE / "build"
    obj_dir.mkdir(exist_ok=True)
    LIB_DIR.mkdir(exist_ok=True)

    def compile_one(src: Path) -> Path:
        obj = obj_dir / (src.stem + ".o")
        cmd = [hipcc, *HIPCC_FLAGS, "-c", str(src), "-o", str(obj)]
        if src.name in NO_SPILL_SOURCES:
            cmd.append("-Rpass-analysis=kernel-resource-usage")
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src.name}:\n{r.stdout}\n{r.stderr}")
        if src.name in NO_SPILL_SOURCES:
            check_no_spills(src.name, r.stderr)
        if verbose:
            print(f"[build] {src.name} -> {obj.name}", flush=True)
        return obj

    with ThreadPoolExecutor(max_workers=min(8, len(sources()))) as ex:
        objs = list(ex.map(compile_one, sources()))
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB_PATH)
    if verbose:
        print(f"[build] linked {LIB_PATH}", flush=True)
    build_torch_library(verbose)
    return LIB_PATH


def build_torch_library(verbose: bool = True) -> Path:
    """csrc/torch_ops.cpp against the installed torch; finds libdsv3fp8.so beside it."""
    import torch
    root = Path(torch.__file__).resolve().parent
    rocm = Path(_hipcc()).resolve().parent.parent
    tmp = TORCH_LIB_PATH.with_suffix(".so.tmp")
    cmd = [shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}", f"-I{root / 'include'}", f"-I{rocm / 'include'}",
           "-isystem/opt/rocm/include", str(TORCH_SRC), "-o", str(tmp), f"-L{root / 'lib'}", "-lc10", "-lc10_hip", "-ltorch_cpu",
           f"-L{LIB_DIR}", "-ldsv3fp8", "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"building {TORCH_LIB_PATH.name} failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, TORCH_LIB_PATH)
    if verbose:
        print(f"[build] linked {TORCH_LIB_PATH}", flush=True)
    return TORCH_LIB_PATH


if __name__ == "__main__":
    build_library()
    sys.exit(0)
