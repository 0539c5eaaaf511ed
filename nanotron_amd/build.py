"""Builds nanotron_amd/libntfp8.so (the C-ABI library of include/ntfp8.h) with hipcc for gfx950.

    python -m nanotron_amd.build               the product library
    python -m nanotron_amd.build --profiling   also the profiling libraries that `bench.py --workload wg-timeline` loads

The libraries are built in-tree so that they travel with the source tree to the GPU box; nothing is
JIT-compiled at import time.

nanotron_amd/_hostcall.so is a CPython extension on top of libntfp8.so: the host side of the hot calls.

Profiling libraries (nanotron_amd/profiling/, loaded by nothing but the benchmark's wg-timeline workload):
libntfp8_stamps.so is the product library with per-workgroup time stamps compiled into the GEMM kernel
(-DNTFP8_STAMPS); the libntfp8_<name>.so beside it carry the same stamps and, for a quick build, only the instantiation
that the forward GEMM launches.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libntfp8.so")
HOSTCALL = os.path.join(HERE, "_hostcall.so")
PROFILING_DIR = os.path.join(HERE, "profiling")
LIB_STAMPS = os.path.join(PROFILING_DIR, "libntfp8_stamps.so")
SOURCES = ["quant.hip", "gemm.hip", "gemm_mid.hip", "gemm_few.hip", "gemm_any.hip", "capi.hip"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
    # packed fp32 VALU ops are kept out of every kernel
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]
# name -> extra defines of gemm.hip
EXPERIMENTS = {"base": []}


def experiment_lib(name: str) -> str:
    return os.path.join(PROFILING_DIR, f"libntfp8_{name}.so")


def _compile(job) -> str:
    src, defines, suffix = job
    obj = os.path.join(CSRC, src.replace(".hip", suffix + ".o"))
    cmd = [HIPCC, *FLAGS, *defines, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _link(out: str, objs) -> None:
    subprocess.check_call([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", out, *objs])


def _build_hostcall() -> str:
    """The host extension: plain C++ against torch's headers, linked to the libntfp8.so beside it."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths, library_paths

    inc = [f"-I{p}" for p in [*include_paths(), "/opt/rocm/include", sysconfig.get_paths()["include"]]]
    libs = [f"-L{p}" for p in library_paths()]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *inc, os.path.join(CSRC, "hostcall.cpp"),
           "-o", HOSTCALL, *libs, "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip", "-ltorch_python", f"-L{HERE}", "-l:libntfp8.so",
           "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed for hostcall.cpp:\n{r.stderr}")
    return HOSTCALL


def build(verbose: bool = True, profiling: bool = False) -> str:
    jobs = [(s, [], "") for s in SOURCES]
    if profiling:
        jobs.append(("gemm.hip", ["-DNTFP8_STAMPS"], "_stamps"))
        jobs += [("gemm.hip", ["-DNTFP8_STAMPS", "-DNTFP8_PROFILE_NARROW", *defs], "_x_" + name)
                 for name, defs in EXPERIMENTS.items()]
    with ThreadPoolExecutor(max_workers=min(len(jobs), 6)) as ex:
        objs = list(ex.map(_compile, jobs))
    plain = objs[:len(SOURCES)]
    _link(LIB, plain)
    built = [LIB, _build_hostcall()]
    if profiling:
        os.makedirs(PROFILING_DIR, exist_ok=True)
        for obj, out in zip(objs[len(SOURCES):], [LIB_STAMPS] + [experiment_lib(n) for n in EXPERIMENTS]):
            _link(out, [obj if o.endswith("gemm.o") else o for o in plain])
            built.append(out)
    if verbose:
        print("built " + " ".join(os.path.relpath(b, HERE) for b in built))
    return LIB


if __name__ == "__main__":
    build(profiling="--profiling" in sys.argv[1:])
