"""Builds libfourbit.so in-tree: hipcc for the gfx950 kernels, g++ for the host packers;
then ``tests/c/abi_gpu``, the GPU tests' native caller of the library's C ABI, and
``libfourbit_trace.so``, a diagnostic copy of the library whose GEMV also records per-wave
phase timestamps (``FB_PHASE_TRACE``; read by ``bench.py --phase-trace``).

Run as ``python -m if_i_could_turn_back_time_amd.build_lib`` (``__graft_entry__.build()``
calls :func:`build`).  Always recompiles.  Objects go to ``_build/`` at the repo root;
the shared library lands next to this file, where ``_capi`` loads it from.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
INCLUDE = ROOT / "include"
BUILD = ROOT / "_build"
LIB = PKG / "libfourbit.so"
TRACE_LIB = PKG / "libfourbit_trace.so"
TORCH_EXT = PKG / "_fourbit_torch.so"
C_TESTS = ROOT / "tests" / "c"
ARCH = "gfx950"

# packed fp32 VALU ops are disabled for every HIP translation unit: a correctness
# precaution for gfx950, where some of their forms have been seen to give wrong results
HIP_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # the GEMV's work counter is a one-lane LDS atomic whose result is used a step later;
    # the wave-aggregating atomic rewrite would wait for it on the spot
    "-mllvm", "-amdgpu-atomic-optimizer-strategy=None",
    # kernel arguments arrive in SGPRs with the wave instead of through a scalar load
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
    "-Wno-unused-command-line-argument",
]
HOST_FLAGS = ["-O3", "-std=c++17", "-fPIC", "-ffp-contract=off", "-Wall"]


def _hipcc() -> str:
    for cand in (shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (ROCm is required to build libfourbit.so)")


def _torch_extension_cmds(obj: Path, out: Path) -> tuple[list[str], list[str]]:
    """The compile and link lines of ``_fourbit_torch``: fourbit_torch.cpp against torch's and
    ROCm's headers, linked to libfourbit.so beside it."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension
    hip = Path(_hipcc()).resolve().parents[1]
    inc = [f"-I{p}" for p in cpp_extension.include_paths()]
    inc += [f"-I{sysconfig.get_paths()['include']}", f"-I{hip / 'include'}", f"-I{INCLUDE}"]
    comp = ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden",
            "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *inc,
            "-c", str(CSRC / "fourbit_torch.cpp"), "-o", str(obj)]
    link = ["g++", "-shared", str(obj), "-o", str(out), f"-L{cpp_extension.library_paths()[0]}",
            "-ltorch_cpu", "-ltorch", "-ltorch_python", "-lc10", "-lc10_hip", f"-L{PKG}",
            "-l:libfourbit.so", "-Wl,-rpath,$ORIGIN"]
    return comp, link


def _run(cmd: list[str]) -> None:
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError(f"build step failed ({r.returncode}): {' '.join(cmd)}")
    # hipcc's host pass warns that it does not know the packed-fp32 feature: harmless
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in r.stderr.splitlines() if noise not in l)
    if err.strip():
        sys.stderr.write(err + "\n")


def build(verbose: bool = False) -> Path:
    BUILD.mkdir(exist_ok=True)
    inc = [f"-I{INCLUDE}", f"-I{CSRC}"]
    host_o = BUILD / "fourbit_host.o"
    gemv_o = BUILD / "fourbit_gemv.o"
    ilp_o = BUILD / "fourbit_gemv_ilp.o"
    gemm_o = BUILD / "fourbit_gemm.o"
    grad_o = BUILD / "fourbit_grad.o"
    pack_o = BUILD / "fourbit_pack.o"
    jenks2_o = BUILD / "fourbit_jenks2.o"
    trace_o = BUILD / "fourbit_gemv_trace.o"
    trace_ilp_o = BUILD / "fourbit_gemv_ilp_trace.o"
    steps = [
        ["g++", *HOST_FLAGS, *inc, "-c", str(CSRC / "fourbit_host.cpp"), "-o", str(host_o)],
        [_hipcc(), *HIP_FLAGS, *inc, "-c", str(CSRC / "fourbit_gemv.hip"), "-o", str(gemv_o)],
        # the batch-1 rotated and the 8-wave short-preload batch-1 kernels: max-ILP scheduling
        # (measured faster for them, and slower for the large layers' kernels)
        [_hipcc(), *HIP_FLAGS, "-mllvm", "-amdgpu-sched-strategy=max-ilp", *inc, "-c",
         str(CSRC / "fourbit_gemv_ilp.hip"), "-o", str(ilp_o)],
        [_hipcc(), *HIP_FLAGS, *inc, "-c", str(CSRC / "fourbit_gemm.hip"), "-o", str(gemm_o)],
        [_hipcc(), *HIP_FLAGS, *inc, "-c", str(CSRC / "fourbit_grad.hip"), "-o", str(grad_o)],
        # the GPU packer must round every fp64 operation as the host packer does
        [_hipcc(), *HIP_FLAGS, "-ffp-contract=off", *inc, "-c", str(CSRC / "fourbit_pack.hip"),
         "-o", str(pack_o)],
        # the two-class Jenks rounds every fp64 operation as its host twin does
        [_hipcc(), *HIP_FLAGS, "-ffp-contract=off", *inc, "-c", str(CSRC / "fourbit_jenks2.hip"),
         "-o", str(jenks2_o)],
        [_hipcc(), *HIP_FLAGS, "-DFB_PHASE_TRACE", *inc, "-c", str(CSRC / "fourbit_gemv.hip"),
         "-o", str(trace_o)],
        [_hipcc(), *HIP_FLAGS, "-mllvm", "-amdgpu-sched-strategy=max-ilp", "-DFB_PHASE_TRACE",
         *inc, "-c", str(CSRC / "fourbit_gemv_ilp.hip"), "-o", str(trace_ilp_o)],
    ]
    ext_tmp = TORCH_EXT.with_suffix(".so.tmp")
    ext_comp, ext_link = _torch_extension_cmds(BUILD / "fourbit_torch.o", ext_tmp)
    steps.append(ext_comp)
    for cmd in steps:
        if verbose:
            print(" ".join(cmd), flush=True)
    # the translation units are independent: compile them side by side
    with ThreadPoolExecutor(max_workers=len(steps)) as ex:
        for f in [ex.submit(_run, cmd) for cmd in steps]:
            f.result()
    for lib, kern_os in ((LIB, (gemv_o, ilp_o)), (TRACE_LIB, (trace_o, trace_ilp_o))):
        tmp = lib.with_suffix(".so.tmp")
        link = [_hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", str(host_o),
                *map(str, kern_os), str(gemm_o), str(grad_o), str(pack_o), str(jenks2_o), "-o", str(tmp), "-lpthread"]
        if verbose:
            print(" ".join(link), flush=True)
        _run(link)
        os.replace(tmp, lib)
    # torch's way in: one native call per forward (needs the library just linked)
    if verbose:
        print(" ".join(ext_link), flush=True)
    _run(ext_link)
    os.replace(ext_tmp, TORCH_EXT)
    # the GPU test suite's native (no Python) caller of the C ABI, linked to the library
    # through a path relative to itself, so that it runs wherever the tree is copied
    caller = [_hipcc(), *HIP_FLAGS, f"-I{INCLUDE}", str(C_TESTS / "abi_gpu.cpp"), "-o",
              str(C_TESTS / "abi_gpu"), f"-L{PKG}", "-l:libfourbit.so",
              "-Wl,-rpath,$ORIGIN/../../if_i_could_turn_back_time_amd"]
    # and the mask of a Jenks split at any position, which the library's entry points do not take
    ties = [_hipcc(), *HIP_FLAGS, "-shared", str(C_TESTS / "jenks2_ties.hip"), "-o",
            str(C_TESTS / "jenks2_ties.so")]
    for cmd in (caller, ties):
        if verbose:
            print(" ".join(cmd), flush=True)
        _run(cmd)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
