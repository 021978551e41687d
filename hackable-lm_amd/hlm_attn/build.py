"""Builds libhlm_attn.so (the HIP kernels + C ABI) for gfx950 with hipcc, the
CPython binding of its forward entry points (_pycall, host code, g++) and the
torch C++ extension of plain eager calls (_torch_fwd, host code).

Both are built in-tree next to this file, so they travel with the source tree
to the machine that runs it.  Usage:  python -m hlm_attn.build  (or build()).
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
import tempfile
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
LIB_PATH = PKG_DIR / "libhlm_attn.so"
SOURCES = ("attn_fwd.hip", "attn_bwd.hip", "attn_bwd_dkdv.hip", "attn_bwd_fused.hip", "qk_norm_rope.hip", "linear_ce.hip", "lm_head_gemm.hip", "residual_norm.hip", "capi.hip")
ARCH = "gfx950"
PYCALL_PATH = PKG_DIR / ("_pycall" + (sysconfig.get_config_var("EXT_SUFFIX") or ".so"))
TORCH_FWD_PATH = PKG_DIR / "_torch_fwd.so"

# -packed-fp32-ops off: no v_pk_{add,mul,fma}_f32 in device code.
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-mllvm", "-amdgpu-mfma-vgpr-form",  # MFMA accumulators in VGPRs: no AGPR copies around the softmax
    "-Wall",
    "-Wno-unused-result",
]
# The attention kernels are scheduled with LLVM's iterative ILP strategy: on
# the MI355X it took 1-5% off the forward and the dQ kernel across the
# benchmark configs (bit-identical results).  The dK/dV kernel keeps the
# default scheduler, which honours its pipelined operand reads within three
# waves per SIMD (iterative ILP spills there); so do the bandwidth-bound
# kernels.
PER_SOURCE_FLAGS = {
    "attn_fwd.hip": ["-mllvm", "-amdgpu-sched-strategy=iterative-ilp"],
    "attn_bwd.hip": ["-mllvm", "-amdgpu-sched-strategy=iterative-ilp"],
}


def hipcc() -> str:
    found = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(found).exists():
        raise RuntimeError("hipcc not found; the HIP attention library needs ROCm's hipcc to build")
    return found


def _run(cmd: list[str]) -> str:
    proc = subprocess.run(cmd, capture_output=True, text=True)
    # hipcc's host pass does not know the device-only feature flag; drop that line.
    noise = "not a recognized feature for this target"
    log = "\n".join(l for l in (proc.stdout + proc.stderr).splitlines() if noise not in l)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed ({proc.returncode}):\n{' '.join(cmd)}\n{log}")
    return log


def build(verbose: bool = False, out: Path | None = None, defines: tuple[str, ...] = ()) -> Path:
    """Compiles every kernel source (one object each, in parallel, with its
    own scheduler flags) and links LIB_PATH (always recompiles).  `out` and
    `defines` (-D flags) build a variant elsewhere, for experiments."""
    target = Path(out) if out is not None else LIB_PATH
    tmp = target.with_suffix(".so.tmp")
    dflags = [f"-D{d}" for d in defines]
    with tempfile.TemporaryDirectory(prefix="hlm_build_") as work:
        objs, cmds = [], []
        for src in SOURCES:
            obj = Path(work) / (Path(src).stem + ".o")
            objs.append(obj)
            cmds.append([hipcc(), *HIPCC_FLAGS, *PER_SOURCE_FLAGS.get(src, []), *dflags, "-c", str(CSRC / src),
                         "-o", str(obj)])
        with ThreadPoolExecutor(max_workers=min(len(cmds), os.cpu_count() or 1)) as pool:
            logs = list(pool.map(_run, cmds))
        logs.append(_run([hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp)]))
    log = "\n".join(l for l in logs if l.strip())
    if verbose and log.strip():
        print(log, file=sys.stderr)
    os.replace(tmp, target)
    if out is None:
        build_pycall()
        build_torch_fwd()
    return target


def build_pycall() -> Path:
    """Compiles csrc/pycall.cpp (CPython API, no device code) into PYCALL_PATH,
    linked against LIB_PATH in the same directory."""
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        raise RuntimeError("no host C++ compiler (g++) for the CPython binding")
    tmp = PYCALL_PATH.with_name(PYCALL_PATH.name + ".tmp")
    _run([cxx, "-O2", "-std=c++17", "-shared", "-fPIC", "-Wall", f"-I{sysconfig.get_paths()['include']}",
          str(CSRC / "pycall.cpp"), f"-L{PKG_DIR}", "-lhlm_attn", "-Wl,-rpath,$ORIGIN", "-o", str(tmp)])
    os.replace(tmp, PYCALL_PATH)
    return PYCALL_PATH



def build_torch_fwd() -> Path:
    """Compiles csrc/torch_fwd.cpp (torch C++ extension, host code only) into
    TORCH_FWD_PATH with g++ and torch's headers, linked against torch and
    against LIB_PATH in the same directory."""
    import torch
    from torch.utils import cpp_extension

    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        raise RuntimeError("no host C++ compiler (g++) for the torch extension")
    abi = int(torch._C._GLIBCXX_USE_CXX11_ABI)
    rocm = Path(hipcc()).resolve().parent.parent
    cmd = [cxx, "-O2", "-std=c++17", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={abi}", "-DTORCH_EXTENSION_NAME=_torch_fwd", "-DTORCH_API_INCLUDE_EXTENSION_H",
           *[f"-I{d}" for d in cpp_extension.include_paths()], f"-I{rocm / 'include'}", f"-I{sysconfig.get_paths()['include']}",
           str(CSRC / "torch_fwd.cpp"),
           *[f"-L{d}" for d in cpp_extension.library_paths()], "-lc10", "-lc10_hip", "-ltorch", "-ltorch_cpu", "-ltorch_python",
           f"-L{PKG_DIR}", "-lhlm_attn", "-Wl,-rpath,$ORIGIN"]
    tmp = TORCH_FWD_PATH.with_name(TORCH_FWD_PATH.name + ".tmp")
    _run([*cmd, "-o", str(tmp)])
    os.replace(tmp, TORCH_FWD_PATH)
    return TORCH_FWD_PATH


if __name__ == "__main__":
    print(build(verbose=True))
