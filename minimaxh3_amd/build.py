"""Build recipe for the native libraries in ``minimaxh3_amd/_lib`` (gfx950 only).

Each ``csrc/*.hip`` file is compiled by hipcc in parallel and the objects are linked into
one shared library, ``libmxf8.so``, exporting the C ABI declared in ``include/mxf8.h``.
``csrc/torch_ops.cpp`` (host code: the hot torch ops over that ABI) becomes
``libmxf8_torch.so``.

    python -m minimaxh3_amd.build            # build (always recompiles)
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
LIBDIR = os.path.join(PKG, "_lib")
LIBNAME = "libmxf8.so"
OPSNAME = "libmxf8_torch.so"
# (source, object name, extra defines); attn_inst.hip is instantiated per (D, out dtype)
SOURCES = [
    ("capi.hip", "capi", []),
    ("quant.hip", "quant", []),
    ("gemm.hip", "gemm", []),
    ("attn.hip", "attn", []),
] + [
    ("attn_inst.hip", f"attn_d{d}_o{o}", [f"-DMXF8_ATTN_D={d}", f"-DMXF8_ATTN_ODT={o}"])
    for d in (128, 64) for o in (0, 1)
]

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fhip-fp32-correctly-rounded-divide-sqrt",
    # keep the compiler from forming packed fp32 VALU ops (v_pk_{add,mul,fma}_f32)
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # start every loop on a 64-byte boundary: where a loop happens to start otherwise moves
    # with unrelated code before it, and the attention loop ran 12% slower from an unlucky
    # start (same instructions, measured on MI355X)
    "-falign-loops=64",
    "-Wno-pass-failed",
]


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(path):
        raise RuntimeError("hipcc not found: the MI355X library cannot be built")
    return path


def _compile(src: str, obj: str, defines) -> None:
    cmd = [hipcc(), *HIPCC_FLAGS, *defines, "-I", os.path.join(ROOT, "include"), "-c", src, "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {os.path.basename(src)}:\n{res.stderr[-8000:]}")


def _run(cmd, what: str) -> None:
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{what} failed:\n{res.stderr[-8000:]}")


def _rocm() -> str:
    return os.path.dirname(os.path.dirname(os.path.realpath(hipcc())))


def _compile_ops(obj: str) -> None:
    import torch
    from torch.utils import cpp_extension

    inc = [*cpp_extension.include_paths(), os.path.join(_rocm(), "include"), sysconfig.get_paths()["include"]]
    _run(["g++", "-std=c++17", "-O2", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *[f"-I{i}" for i in inc],
          "-c", os.path.join(CSRC, "torch_ops.cpp"), "-o", obj], "g++ torch_ops.cpp")


def _link_ops(obj: str) -> None:
    from torch.utils import cpp_extension

    out = os.path.join(LIBDIR, OPSNAME)
    libs = [f"-L{p}" for p in (*cpp_extension.library_paths(), os.path.join(_rocm(), "lib"), LIBDIR)]
    _run(["g++", "-shared", "-o", out + ".tmp", obj, *libs, f"-l:{LIBNAME}", "-ltorch", "-ltorch_cpu", "-ltorch_python",
          "-lc10", "-lc10_hip", "-lamdhip64", "-Wl,-rpath,$ORIGIN"], "link of the torch ops")
    os.replace(out + ".tmp", out)


def build(verbose: bool = True) -> str:
    """Compile every HIP source for gfx950 and link libmxf8.so (returns its path), then the
    torch ops over it."""
    os.makedirs(LIBDIR, exist_ok=True)
    objdir = os.path.join(LIBDIR, "obj")
    os.makedirs(objdir, exist_ok=True)
    jobs = []
    for name, objname, defines in SOURCES:
        jobs.append((os.path.join(CSRC, name), os.path.join(objdir, objname + ".o"), defines))
    workers = min(len(jobs), max(1, min(8, os.cpu_count() or 1)))
    with ThreadPoolExecutor(max_workers=workers) as ex:
        futs = [ex.submit(_compile, s, o, d) for s, o, d in jobs]
        ops_obj = os.path.join(objdir, "torch_ops.o")
        futs.append(ex.submit(_compile_ops, ops_obj))
        for f in futs:
            f.result()
    out = os.path.join(LIBDIR, LIBNAME)
    tmp = out + ".tmp"
    cmd = [hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *[o for _, o, _ in jobs]]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr[-8000:]}")
    os.replace(tmp, out)
    _link_ops(ops_obj)
    if verbose:
        print(f"[minimaxh3_amd] built {out} and {OPSNAME}")
    return out


if __name__ == "__main__":
    build()
    sys.exit(0)
