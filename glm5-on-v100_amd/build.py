"""Builds libmi355_dsa.so (all HIP kernels + the C ABI) for gfx950, in-tree.

Usage: python glm5-on-v100_amd/build.py   (or __graft_entry__.build())

Each csrc/*.hip is compiled to an object in _build/ (in parallel), then the
objects are linked into <package>/libmi355_dsa.so.  Kernels that rely on a
property of the generated code are checked for it (check_kernels).  hipcc cross-compiles
gfx950 code without a GPU.
"""
from __future__ import annotations

import concurrent.futures as cf
import glob
import os
import re
import shutil
import subprocess
import sys

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG_DIR, "csrc")
BUILD_DIR = os.path.join(PKG_DIR, "_build")
LIB_NAME = "libmi355_dsa.so"
LIB_PATH = os.path.join(PKG_DIR, LIB_NAME)
ARCH = "gfx950"


def hipcc() -> str:
    p = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(p):
        raise RuntimeError("hipcc not found; the HIP toolchain is required")
    return p


def compile_flags() -> list[str]:
    return [
        f"--offload-arch={ARCH}",
        "-O3",
        "-std=c++17",
        "-fPIC",
        "-Wall",
        "-Wno-unused-function",
        # packed fp32 VALU forms are kept out of generated code on purpose
        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
        "-I", os.path.join(PKG_DIR, "..", "include"),
    ]


# Kernels of each source whose generated code the build checks (check_kernels):
# those that hold values in accumulation registers named in inline asm, which
# the compiler does not know to be in use.
OWN_AGPRS = {"sparse_mla.hip": ["mla_hw_f16_kernel"]}
# Kernels that must not spill: a reload in a loop waits for all of the wave's
# memory operations, gathers in flight included.
NO_SPILLS = {"sparse_mla.hip": ["sparse_mla_prefill_fp8_ws_kernel", "sparse_mla_few_kernelILb0E"],
             "varlen_attn.hip": [f"varlen_attn_ring_kernelILb{t}ELi{d}E" for t in (0, 1)
                                 for d in (192, 128, 64)]}


def _body(asm: str, kernel: str) -> tuple[str, list[str]]:
    """The symbol and the assembly lines of the one kernel whose name holds `kernel`."""
    names = [n for n in re.findall(r"^(_Z\w+):", asm, re.M)
             if kernel in n and f"\n\t.amdhsa_kernel {n}\n" in asm]
    if len(names) != 1:
        raise RuntimeError(f"{kernel}: {len(names)} kernels of that name in the assembly")
    start = asm.index(f"\n{names[0]}:")
    return names[0], asm[start:asm.index(".Lfunc_end", start)].split("\n")


def _usage(asm: str, symbol: str, key: str) -> int:
    """An entry of the kernel's metadata (".vgpr_spill_count" and the like)."""
    for block in asm[asm.index("amdhsa.kernels:"):].split("\n  - ")[1:]:
        if re.search(rf"\.name:\s+{re.escape(symbol)}\s", block):
            return int(re.search(rf"{re.escape(key)}:\s+(\d+)", block).group(1))
    raise RuntimeError(f"{symbol}: no metadata")


def check_kernels(asm: str, own_agprs: list[str], no_spills: list[str] = []) -> None:
    """Raises unless no kernel of either list spills or uses scratch memory, and
    every kernel of `own_agprs` is as its inline asm needs it: at most 256 other
    registers, and no instruction that the compiler placed names an accumulation
    register."""
    for kernel in [*own_agprs, *no_spills]:
        symbol, lines = _body(asm, kernel)
        used = {k: _usage(asm, symbol, k) for k in
                (".vgpr_spill_count", ".sgpr_spill_count", ".private_segment_fixed_size")}
        if any(used.values()):
            raise RuntimeError(f"{kernel}: spills: {used}")
        if kernel not in own_agprs:
            continue
        if _usage(asm, symbol, ".vgpr_count") - _usage(asm, symbol, ".agpr_count") > 256:
            raise RuntimeError(f"{kernel}: too many registers")
        in_asm = False
        for line in lines:
            if "#ASMSTART" in line or "#ASMEND" in line:
                in_asm = "#ASMSTART" in line
                continue
            code = line.split(";")[0].strip()
            if not in_asm and re.search(r"\s(?:\S*,\s*)*a(?:\d+|\[\d+:\d+\])", code):
                raise RuntimeError(f"{kernel}: the compiler uses an accumulation register: {code}")


def _compile(src: str) -> str:
    name = os.path.basename(src)
    obj = os.path.join(BUILD_DIR, name.replace(".hip", ".o"))
    cmd = [hipcc(), *compile_flags(), "-c", src, "-o", obj]
    checked = name in OWN_AGPRS or name in NO_SPILLS
    if checked:  # the assembly that the object is made from, beside it
        cmd.append("-save-temps=obj")
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stdout}\n{r.stderr}")
    if checked:
        with open(asm_path(name)) as f:
            check_kernels(f.read(), OWN_AGPRS.get(name, []), NO_SPILLS.get(name, []))
    return obj


def asm_path(name: str) -> str:
    """Where the build leaves the device assembly of a checked source."""
    return os.path.join(BUILD_DIR, name.replace(".hip", f"-hip-amdgcn-amd-amdhsa-{ARCH}.s"))


TESTKIT_SRC = os.path.join(PKG_DIR, "..", "tests", "hip", "quant_exhaustive.hip")
TESTKIT_LIB = os.path.join(PKG_DIR, "..", "tests", "hip", "libdsa_testkit.so")


def build_testkit(verbose: bool = True) -> str:
    """Builds the test-only kernels (tests/hip/*.hip) into
    tests/hip/libdsa_testkit.so; the product library does not contain them."""
    tmp = TESTKIT_LIB + ".tmp"
    cmd = [hipcc(), *compile_flags(), "-shared", TESTKIT_SRC, "-o", tmp]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {TESTKIT_SRC}:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, TESTKIT_LIB)
    if verbose:
        print(f"built {os.path.normpath(TESTKIT_LIB)}", flush=True)
    return TESTKIT_LIB


def build(verbose: bool = True) -> str:
    os.makedirs(BUILD_DIR, exist_ok=True)
    sources = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    if not sources:
        raise RuntimeError("no HIP sources found")
    jobs = min(len(sources), max(1, min(8, os.cpu_count() or 1)))
    with cf.ThreadPoolExecutor(jobs) as ex:
        objs = list(ex.map(_compile, sources))
    tmp = LIB_PATH + ".tmp"
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB_PATH)
    if verbose:
        print(f"built {LIB_PATH} from {len(sources)} sources", flush=True)
    return LIB_PATH


if __name__ == "__main__":
    build()
    build_testkit()
    sys.exit(0)
