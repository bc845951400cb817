"""Build recipe for libfarope.so (hand-written gfx950 HIP kernels + C ABI) and
libfarope_torch.so (the torch ops' GPU kernels over it, host code).

Compiles every HIP translation unit under csrc/ with hipcc for gfx950 (in
parallel), then links the shared libraries next to this file, where
``_lib.py`` loads them.  Runs on a machine without a GPU: hipcc
cross-compiles.  ``python -m triton_fused_rope_flash_attn_amd.build``.
"""
from __future__ import annotations

import concurrent.futures as _cf
import os
import shutil
import subprocess
import sys
import tempfile

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
REPO_DIR = os.path.dirname(PKG_DIR)
CSRC = os.path.join(PKG_DIR, "csrc")
INCLUDE = os.path.join(REPO_DIR, "include")
LIB_NAME = "libfarope.so"
LIB_PATH = os.path.join(PKG_DIR, LIB_NAME)
SOURCES = ["api.hip", "fwd.hip", "fwd_plane.hip", "fwd_stream.hip", "bwd.hip", "bwd_fused.hip", "bwd_keys.hip", "bwd_ds.hip", "bwd_stream.hip", "short.hip", "tail.hip"]
# Per-file code generation options.  fwd_plane.hip keeps its MFMA results in
# VGPRs (they feed the softmax VALU directly) and its resident operand
# fragments in AGPRs.
EXTRA_FLAGS = {"fwd_plane.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"]}
ARCH = "gfx950"
OPS_SOURCE = "torch_ops.cpp"
OPS_PATH = os.path.join(PKG_DIR, "libfarope_torch.so")


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found: the ROCm toolchain is required to build libfarope.so")


def compile_flags() -> list[str]:
    return [
        f"--offload-arch={ARCH}",
        "-O3",
        "-std=c++17",
        "-fPIC",
        "-ffp-contract=fast",
        # The kernels never depend on NaN semantics (masked logits are -inf):
        # with IEEE mode off, fmax needs no operand canonicalization.
        "-fno-honor-nans",
        "-mno-amdgpu-ieee",
        "-mcode-object-version=5",
        # Packed-fp32 VALU forms are kept out of the generated code.
        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
        f"-I{INCLUDE}",
        f"-I{CSRC}",
        "-Wno-unused-result",
    ]


def _run(cmd: list[str]) -> None:
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(
        ln for ln in res.stdout.splitlines() if "packed-fp32-ops" not in ln
    )
    if res.returncode != 0:
        raise RuntimeError(f"command failed ({res.returncode}): {' '.join(cmd)}\n{out}")


def ops_commands(obj: str, out: str) -> list[list[str]]:
    """Compile and link commands of the torch ops library (host code against
    torch's headers; it finds libfarope.so next to itself)."""
    import torch

    tdir = os.path.dirname(torch.__file__)
    hipcc = _hipcc()
    rocm_inc = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(hipcc))), "include")
    compile_ = [hipcc, "-x", "c++", "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
                f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
                f"-I{INCLUDE}", f"-I{tdir}/include", f"-I{tdir}/include/torch/csrc/api/include", f"-I{rocm_inc}",
                "-Wno-deprecated-declarations", "-c", os.path.join(CSRC, OPS_SOURCE), "-o", obj]
    link = [hipcc, "-shared", "-fPIC", obj, "-o", out, f"-L{PKG_DIR}", "-l:" + LIB_NAME, f"-L{tdir}/lib",
            "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch", "-Wl,-rpath,$ORIGIN"]
    return [compile_, link]


def build(verbose: bool = False, jobs: int | None = None) -> str:
    """Compile and link libfarope.so and libfarope_torch.so; returns the former's path."""
    hipcc = _hipcc()
    flags = compile_flags()
    tmp = tempfile.mkdtemp(prefix="farope_build_")
    try:
        objs = []
        cmds = []
        for src in SOURCES:
            obj = os.path.join(tmp, src.replace(".hip", ".o"))
            objs.append(obj)
            cmds.append([hipcc, *flags, *EXTRA_FLAGS.get(src, []), "-c", os.path.join(CSRC, src), "-o", obj])
        ops_obj, ops_out = os.path.join(tmp, "torch_ops.o"), OPS_PATH + ".tmp"
        ops_compile, ops_link = ops_commands(ops_obj, ops_out)
        cmds.append(ops_compile)
        jobs = jobs or min(len(cmds), os.cpu_count() or 1, 16)
        with _cf.ThreadPoolExecutor(max_workers=jobs) as ex:
            for cmd, fut in zip(cmds, [ex.submit(_run, c) for c in cmds]):
                if verbose:
                    print(" ".join(cmd), flush=True)
                fut.result()
        out_tmp = LIB_PATH + ".tmp"
        _run([hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", out_tmp])
        os.replace(out_tmp, LIB_PATH)
        _run(ops_link)
        os.replace(ops_out, OPS_PATH)
    finally:
        shutil.rmtree(tmp, ignore_errors=True)
    if verbose:
        print(f"built {LIB_PATH} and {OPS_PATH}", flush=True)
    return LIB_PATH


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
