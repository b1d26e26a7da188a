"""What the attention's code arithmetic (attn_codes_tile) needs of the compiled kernels: nothing but its
FMAs runs while fp32 denormal results are flushed, and its byte writes are followed by wait states.  Both
hold by construction where each lies inside one asm statement, in which the compiler places nothing."""
import os
import re
import subprocess

import pytest

from minimaxh3_amd import build

FLUSH, KEEP = (f"s_setreg_imm32_b32 hwreg(HW_REG_MODE, 4, 2), {bits}" for bits in (1, 3))


@pytest.fixture(scope="module")
def asm(tmp_path_factory):
    out = tmp_path_factory.mktemp("asm") / "attn.s"
    res = subprocess.run([build.hipcc(), *build.HIPCC_FLAGS, "-DMXF8_ATTN_D=64", "-DMXF8_ATTN_ODT=0", "-I",
                          os.path.join(build.ROOT, "include"), "--offload-device-only", "-S", "-o", str(out),
                          os.path.join(build.CSRC, "attn_inst.hip")], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-4000:]
    return out.read_text()


def _statements(asm):
    """Instructions of every asm statement, and those outside."""
    parts = re.split(r";;?#ASMSTART\n(.*?);;?#ASMEND\n", asm, flags=re.S)

    def ins(text):
        return [line.strip() for line in text.splitlines() if line.strip()[:1].islower()]

    return [ins(p) for p in parts[1::2]], [i for p in parts[::2] for i in ins(p)]


def test_flush_window_holds_only_the_fmas(asm):
    stmts, outside = _statements(asm)
    assert not any(i in (FLUSH, KEEP) for i in outside)
    windows = [s for s in stmts if FLUSH in s or KEEP in s]
    assert len(windows) >= 24  # two per tile of every kernel without the repair
    for s in windows:
        assert s[0] == FLUSH and s.count(FLUSH) == s.count(KEEP) == 1
        body = s[1:s.index(KEEP)]
        assert len(body) == 32 and all(re.fullmatch(r"v_fma_f32 v\d+, v\d+, v\d+, v\d+ clamp", i) for i in body)


def test_byte_writes_end_with_wait_states(asm):
    """One wait state between two writes of a word, two from the last write to a matrix product."""
    stmts, _ = _statements(asm)  # (outside them the compiler minds its own)
    blocks = [s for s in stmts if any("sdwa" in i for i in s)]
    assert blocks
    for s in blocks:
        assert s[-1] == "s_nop 1"
        dst = [i.split()[1] for i in s[:-1] if i.startswith("v_mul")]
        assert all(a != b for a, b in zip(dst, dst[1:]))


def test_no_kernel_spills(asm):
    spills = re.findall(r"\.vgpr_spill_count:\s+(\d+)", asm)
    assert spills and set(spills) == {"0"}
