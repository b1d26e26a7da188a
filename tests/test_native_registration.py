"""The hot ops' native kernels are in the dispatcher once the package is imported, before any call
(no GPU needed): registering them under another thread's call would change a table that the
dispatcher reads without a lock."""
import subprocess
import sys

import pytest

OPS = ("quant_rows", "adaln_quant_rows", "gemm_rowwise", "lora_down", "attn_quant_kv", "attn_fwd_q")


def _python(code):
    res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-4000:]
    return res.stdout.split()


@pytest.mark.parametrize("module", ["minimaxh3_amd.ops", "minimaxh3_amd.kernels.fp8_linear",
                                    "minimaxh3_amd.kernels.fp8_attention"])
def test_import_registers_the_native_kernels(module):
    out = _python(f"""
import torch, {module}
for op in {OPS}:
    for key in ("CUDA", "AutogradCUDA"):
        print(torch._C._dispatch_has_kernel_for_dispatch_key("mxf8::" + op, key))
print(not torch.cuda.is_initialized())
""")
    assert out == ["True"] * (2 * len(OPS) + 1)


@pytest.mark.parametrize("content", [None, "not a library"])
def test_import_without_a_usable_library(content, tmp_path):
    """The build recipe and CPU-only code import the package without it, and calls say so."""
    path = tmp_path / "libmxf8_torch.so"
    if content is not None:
        path.write_text(content)
    out = _python(f"""
import minimaxh3_amd._native as N
N._OPS_PATH = {str(path)!r}
import minimaxh3_amd.ops, torch
try:
    N.load_ops()
except (OSError, RuntimeError) as e:
    print("raises")
try:
    minimaxh3_amd.ops.quant_rows(torch.zeros(2, 16))
except ValueError as e:
    print("refuses")
""")
    assert out == ["raises", "refuses"]
