"""Builds dax_amd/lib/libdaxq.so from dax_amd/csrc with hipcc for gfx950.

Cross-compiles without a GPU.  Used by ``__graft_entry__.build()``; the tests, the
smoke run and the benchmark load the library that is already there.
"""
from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIBDIR, "libdaxq.so")
ROOT = os.path.dirname(HERE)
TORCH_LIB = os.path.join(LIBDIR, "_daxq_torch.so")
MFMA_RATE = os.path.join(ROOT, "bench", "mfma_rate")
SOURCES = ["capi.hip", "quant_rows.hip", "quant_blocks.hip", "fused_rows.hip", "per_tensor.hip", "gemm_w8a8.hip", "gemm_rows.hip", "gemm_few.hip", "gemm_tile256.hip", "gemm_tile_fp8.hip", "gemm_tile_fit.hip", "gemm_tile_fit_fp8.hip"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fno-fast-math",
    # packed-FP32 VALU forms are kept out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-command-line-argument",
]


# Every source but the fused producers is compiled without floating-point contraction: a multiply followed by an
# add (INT8 / FP8 epilogues: scale, scale, bias) or by a narrowing convert (fp16 outputs) must round once per
# operation, as the reference's op sequence does; contraction turns them into an fma or a mixed-precision fma with a
# single rounding.  fused_rows.hip (LayerNorm / GELU statistics, compared at a stated tolerance) keeps its fmas.
NO_CONTRACT = {"quant_rows.hip", "quant_blocks.hip", "per_tensor.hip", "gemm_w8a8.hip", "gemm_rows.hip", "gemm_few.hip", "gemm_tile256.hip", "gemm_tile_fp8.hip", "gemm_tile_fit.hip", "gemm_tile_fit_fp8.hip"}


def _compile(src: str, verbose: bool) -> str:
    obj = os.path.join(LIBDIR, os.path.splitext(src)[0] + ".o")
    extra = ["-ffp-contract=off"] if src in NO_CONTRACT else []
    cmd = [HIPCC, *FLAGS, *extra, "-c", os.path.join(CSRC, src), "-o", obj]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l and l.strip())
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{err}")
    if err and verbose:
        print(err, file=sys.stderr)
    return obj


def _compile_torch_entry(verbose: bool) -> str:
    """torch_linear.cpp (host code against torch's headers), linked once libdaxq.so is there."""
    import torch
    from torch.utils.cpp_extension import include_paths

    obj = os.path.join(LIBDIR, "torch_linear.o")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-Wall", "-DUSE_ROCM=1", "-D__HIP_PLATFORM_AMD__=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *(f"-isystem{d}" for d in (*include_paths("cuda"), sysconfig.get_paths()["include"])),
           "-c", os.path.join(CSRC, "torch_linear.cpp"), "-o", obj]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed on torch_linear.cpp:\n{r.stderr}")
    return obj


def _link_torch_entry(obj: str, verbose: bool) -> None:
    import torch

    # libdaxq.so beside it is the library that ctypes loads, too; torch's libraries are loaded before this one
    cmd = ["g++", "-shared", "-o", TORCH_LIB, obj, "-L" + LIBDIR, "-l:libdaxq.so", "-Wl,-rpath,$ORIGIN",
           "-L" + os.path.join(os.path.dirname(torch.__file__), "lib"), "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python"]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link of _daxq_torch.so failed:\n{r.stderr}")


def build(verbose: bool = False) -> str:
    os.makedirs(LIBDIR, exist_ok=True)
    with ThreadPoolExecutor(max_workers=len(SOURCES) + 1) as ex:
        entry = ex.submit(_compile_torch_entry, verbose)
        objs = list(ex.map(lambda s: _compile(s, verbose), SOURCES))
        entry = entry.result()
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB, *objs]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    _link_torch_entry(entry, verbose)
    # stand-alone microbenchmark behind bench.py's sustained-MFMA-rate figure
    cmd = [HIPCC, *FLAGS, os.path.join(ROOT, "bench", "mfma_rate.hip"), "-o", MFMA_RATE]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on mfma_rate.hip:\n{r.stderr}")
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
