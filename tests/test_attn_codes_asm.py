"""What the attention's code arithmetic (attn_codes_tile) needs of the compiled kernels: nothing but its
FMAs runs while fp32 denormal results are flushed, and its byte writes are followed by wait states."""
import os
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from minimaxh3_amd import build

FLUSH, KEEP = (f"s_setreg_imm32_b32 hwreg(HW_REG_MODE, 4, 2), {bits}" for bits in (1, 3))
BUILDS = [defines for src, _, defines in build.SOURCES if src == "attn_inst.hip"]


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    """The assembly of every attention object of the build, by its defines."""
    tmp = tmp_path_factory.mktemp("asm")

    def compile_(i):
        out = tmp / f"{i}.s"
        res = subprocess.run([build.hipcc(), *build.HIPCC_FLAGS, *BUILDS[i], "-I", os.path.join(build.ROOT, "include"),
                              "--offload-device-only", "-S", "-o", str(out), os.path.join(build.CSRC, "attn_inst.hip")],
                             capture_output=True, text=True)
        assert res.returncode == 0, res.stderr[-4000:]
        return out.read_text()

    with ThreadPoolExecutor(max_workers=4) as ex:
        return list(ex.map(compile_, range(len(BUILDS))))


def _instructions(text):
    """Instructions and labels (a label ends with a colon), without the assembler's comments."""
    lines = (line.split(";")[0].strip() for line in text.splitlines())
    return [line for line in lines if line[:1].islower() or re.fullmatch(r"\.LBB\w+:", line)]


@pytest.mark.parametrize("which", range(len(BUILDS)), ids=[" ".join(d) for d in BUILDS])
def test_flush_window_holds_only_the_fmas(assembly, which):
    ins = _instructions(assembly[which])
    start = [i for i, s in enumerate(ins) if s == FLUSH]
    assert len(start) >= 12 and sum(s == KEEP for s in ins) == len(start)  # every kernel without the repair
    for a in start:
        body = [s for s in ins[a + 1:ins.index(KEEP, a)] if not s.startswith("s_nop")]
        assert len(body) == 64 and all(re.fullmatch(r"v_fma_f32 v\d+, v\d+, v\d+, v\d+ clamp", s) for s in body), body


@pytest.mark.parametrize("which", range(len(BUILDS)), ids=[" ".join(d) for d in BUILDS])
def test_byte_writes_end_with_wait_states(assembly, which):
    """One wait state between two writes of a word, two from the last write to a matrix product, inside
    the asm statement, where the compiler places nothing."""
    stmts = [_instructions(s) for s in re.findall(r";;?#ASMSTART\n(.*?);;?#ASMEND\n", assembly[which], flags=re.S)]
    blocks = [s for s in stmts if any("sdwa" in i for i in s)]  # (outside them the compiler minds its own)
    assert len(blocks) >= 48
    for s in blocks:
        assert s[-1] == "s_nop 1"
        dst = [i.split()[1] for i in s[:-1]]
        assert all(a != b for a, b in zip(dst, dst[1:]))


@pytest.mark.parametrize("which", range(len(BUILDS)), ids=[" ".join(d) for d in BUILDS])
def test_registers(assembly, which):
    """No kernel spills, and at D = 64 three waves per SIMD stay resident without the repair (168 of 512
    registers), but for the mask with a bias."""
    spills = re.findall(r"\.vgpr_spill_count:\s+(\d+)", assembly[which])
    assert spills and set(spills) == {"0"}
    if "-DMXF8_ATTN_D=64" in BUILDS[which]:
        kernels = re.findall(r"\.name:\s+(\S*attn_fwd_kernelILi64ELb(\d)ELb(\d)ELb0E\S*).*?\.vgpr_count:\s+(\d+)",
                             assembly[which], flags=re.S)
        assert len(kernels) == 8
        assert all(int(n) <= 168 for _, mask, bias, n in kernels if mask + bias != "11")
