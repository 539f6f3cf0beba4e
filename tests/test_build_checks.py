"""The build's checks of generated code (build.check_kernels), on the assembly
of this tree and on the same text with one property broken."""
import importlib.util
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NAME = "sparse_mla.hip"
KERNEL = "mla_hw_f16_kernel"


@pytest.fixture(scope="module")
def build():
    spec = importlib.util.spec_from_file_location(
        "pkg_build", os.path.join(ROOT, "glm5-on-v100_amd", "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


@pytest.fixture(scope="module")
def asm(build):
    src = os.path.join(build.CSRC, NAME)
    path = build.asm_path(NAME)
    if not os.path.exists(path) or os.path.getmtime(path) < os.path.getmtime(src):
        os.makedirs(build.BUILD_DIR, exist_ok=True)
        build._compile(src)
    with open(path) as f:
        return f.read()


def test_this_tree_passes(build, asm):
    build.check_kernels(asm, build.OWN_AGPRS[NAME], build.NO_SPILLS[NAME])


@pytest.mark.parametrize("line", ["v_accvgpr_write_b32 a7, v3", "v_accvgpr_read_b32 v3, a255",
                                  "v_mfma_f32_16x16x32_f16 a[0:3], v[0:3], v[4:7], 0"])
def test_an_accumulation_register_of_the_compilers(build, asm, line):
    symbol, _ = build._body(asm, KERNEL)
    start = asm.index(f"\n{symbol}:")
    end = asm.index("s_endpgm", start)
    with pytest.raises(RuntimeError, match="accumulation register"):
        build.check_kernels(asm[:end] + line + "\n\t" + asm[end:], [KERNEL])
    # the same line inside an asm block is the kernel's own
    build.check_kernels(asm[:end] + f";;#ASMSTART\n\t{line}\n\t;;#ASMEND\n\t" + asm[end:], [KERNEL])


@pytest.mark.parametrize("key", [".vgpr_spill_count", ".sgpr_spill_count",
                                 ".private_segment_fixed_size"])
@pytest.mark.parametrize("own,none", [([KERNEL], []), ([], [KERNEL])], ids=["own", "none"])
def test_spills_and_scratch(build, asm, key, own, none):
    symbol, _ = build._body(asm, KERNEL)
    head, _, meta = asm.partition("amdhsa.kernels:")
    blocks = meta.split("\n  - ")
    i = next(i for i, b in enumerate(blocks) if re.search(rf"\.name:\s+{symbol}\s", b))
    blocks[i] = re.sub(rf"{re.escape(key)}:(\s+)\d+", rf"{key}:\g<1>4", blocks[i])
    with pytest.raises(RuntimeError, match="spills"):
        build.check_kernels(head + "amdhsa.kernels:" + "\n  - ".join(blocks), own, none)


def test_a_missing_kernel(build, asm):
    with pytest.raises(RuntimeError, match="0 kernels"):
        build.check_kernels(asm, ["no_such_kernel"])
