"""Build the HIP library (gfx950) and the host test shim, in-tree.

``libdetllm_hip.so``      — every kernel + the extern "C" boundary
                            (declared in include/detllm_hip.h);
``_native.so``            — the entry points as Python callables and torch
                            operators (csrc/torch_binding.cpp);
``libdetllm_intops_host.so`` — intops.h compiled for the CPU, used by the
                            CPU test suite to check the integer routines the
                            kernels share.

hipcc compiles each .hip translation unit to an object in parallel, then
links one shared library. Flags: gfx950 only; packed-fp32 instruction
selection disabled (no float arithmetic is used, the flag guards against
compiler-generated v_pk_*_f32).
"""

from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess

PKG = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG, "csrc")
BUILD = os.path.join(os.path.dirname(PKG), "_build")
LIB = os.path.join(PKG, "libdetllm_hip.so")
NATIVE = os.path.join(PKG, "_native.so")
HOST_LIB = os.path.join(PKG, "libdetllm_intops_host.so")
HIP_SOURCES = ("gemm.hip", "rowops.hip", "attention.hip")
ARCH = "gfx950"
HIPCC_FLAGS = ["-O3", "-std=c++17", f"--offload-arch={ARCH}", "-fPIC",
               "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
               "-Wno-unused-result"]


def _hipcc() -> str:
    for cand in (shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found: the ROCm toolchain is required to build the library")


def _run(cmd):
    p = subprocess.run(cmd, capture_output=True, text=True)
    if p.returncode != 0:
        raise RuntimeError(f"build failed: {' '.join(cmd)}\n{p.stdout}\n{p.stderr}")
    return p


def build(verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    hipcc = _hipcc()
    objs = []
    jobs = []
    for src in HIP_SOURCES:
        obj = os.path.join(BUILD, src.replace(".hip", ".o"))
        objs.append(obj)
        jobs.append([hipcc, *HIPCC_FLAGS, "-c", os.path.join(CSRC, src), "-o", obj])
    with cf.ThreadPoolExecutor(max_workers=min(8, len(jobs))) as ex:
        for p in ex.map(_run, jobs):
            if verbose and p.stderr:
                print(p.stderr)
    tmp = LIB + ".tmp"
    _run([hipcc, "-shared", f"--offload-arch={ARCH}", "-fPIC", *objs, "-o", tmp])
    os.replace(tmp, LIB)
    build_native()
    build_host_shim()
    return LIB


def build_native() -> str:
    """The Python / torch binding, linked against the library just built
    (found next to it) and torch's own libraries (loaded by ``import torch``)."""
    import sysconfig

    import torch
    gxx = shutil.which("g++") or "g++"
    root = os.path.dirname(torch.__file__)
    inc = [os.path.join(root, "include"),
           os.path.join(root, "include", "torch", "csrc", "api", "include"),
           sysconfig.get_paths()["include"],
           os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include")]
    tmp = NATIVE + ".tmp"
    _run([gxx, "-O2", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
          *(f"-I{d}" for d in inc), os.path.join(CSRC, "torch_binding.cpp"), "-o", tmp,
          "-L" + os.path.join(root, "lib"), "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip",
          "-L" + PKG, "-l:libdetllm_hip.so", "-Wl,-rpath,$ORIGIN"])
    os.replace(tmp, NATIVE)
    return NATIVE


def build_host_shim() -> str:
    gxx = shutil.which("g++") or "g++"
    tmp = HOST_LIB + ".tmp"
    _run([gxx, "-O2", "-std=c++17", "-shared", "-fPIC", "-I", CSRC,
          os.path.join(CSRC, "intops_host.cpp"), "-o", tmp])
    os.replace(tmp, HOST_LIB)
    return HOST_LIB


if __name__ == "__main__":
    print(build(verbose=True))
