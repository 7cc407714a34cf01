"""Builds libsqattn_hip.so (the product: everything include/sqattn.h declares) and libsqattn_probe.so (a measurement
aid the benchmark loads) in-tree with plain hipcc for gfx950 (no torch extension, no pybind)."""
from __future__ import annotations

import os
import subprocess
import sys

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG_DIR, "csrc")
INCLUDE = os.path.join(os.path.dirname(PKG_DIR), "include")
LIB_PATH = os.path.join(PKG_DIR, "libsqattn_hip.so")
PROBE_LIB_PATH = os.path.join(PKG_DIR, "libsqattn_probe.so")
HOST_CALLS_PATH = os.path.join(PKG_DIR, "_host_calls.so")   # host code on torch's tensors, no GPU code in it
HOST_CALLS_SOURCE = "host_calls.cpp"
SOURCES = ["capi.hip", "decode_gfx950.hip", "prefill_gfx950.hip", "kmeans_gfx950.hip", "prepass_gfx950.hip", "kvcache_gfx950.hip", "layer_gfx950.hip", "linear_gfx950.hip", "gemm_gfx950.hip", "calib_gfx950.hip"]
PROBE_SOURCES = ["capi.hip", "probe_gfx950.hip"]   # its own copy of the error string and the tensor checks

HIPCC_FLAGS = [
    "-O3", "-std=c++17", "--offload-arch=gfx950", "-fPIC", "-shared",
    # keep the compiler from forming packed-fp32 VALU ops
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


# Per-source flags.  The k-means assign kernel reads its MFMA results with the vector ALU right away (arg-max): the MFMAs
# are kept in their VGPR form there, otherwise every score passes through a v_accvgpr_read first.
# The 4-wave prefill workgroups may use 512 registers per lane; in the other form their score accumulators move to AGPRs and back.
SOURCE_FLAGS = {"kmeans_gfx950.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"], "prefill_gfx950.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
                "gemm_gfx950.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"]}


def host_calls_command() -> list:
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths

    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    return [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f'-DSQ_TORCH_VERSION="{torch.__version__}"', "-I", sysconfig.get_paths()["include"], "-I", INCLUDE,
            *(x for p in include_paths() for x in ("-isystem", p)), os.path.join(CSRC, HOST_CALLS_SOURCE),
            "-L", torch_lib, "-ltorch_python", "-ltorch_cpu", "-ltorch", "-lc10", "-o", HOST_CALLS_PATH]


def build(verbose: bool = True, extra_flags=()) -> str:
    """Compile every HIP source (in parallel, one object each) and link the two shared libraries, and the host calls beside them;
    returns the path of the product library.  Always recompiles; a listed source that is missing is an error."""
    import tempfile

    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    srcs = list(dict.fromkeys(SOURCES + PROBE_SOURCES))
    missing = [s for s in srcs + [HOST_CALLS_SOURCE] if not os.path.exists(os.path.join(CSRC, s))]
    if missing:
        raise FileNotFoundError(f"HIP sources missing from {CSRC}: {', '.join(missing)}")
    compile_flags = [f for f in HIPCC_FLAGS if f != "-shared"]
    with tempfile.TemporaryDirectory(prefix="sqattn_build_") as tmp:
        cmd = host_calls_command()
        if verbose:
            print(" ".join(cmd), flush=True)
        jobs = [(cmd, HOST_CALLS_PATH, subprocess.Popen(cmd))]
        for s in srcs:
            obj = os.path.join(tmp, s.replace(".hip", ".o"))
            cmd = [hipcc, *compile_flags, *SOURCE_FLAGS.get(s, []), *extra_flags, "-I", INCLUDE, "-I", CSRC, "-c", os.path.join(CSRC, s), "-o", obj]
            if verbose:
                print(" ".join(cmd), flush=True)
            jobs.append((cmd, obj, subprocess.Popen(cmd)))
        for cmd, obj, proc in jobs:
            if proc.wait() != 0:
                raise subprocess.CalledProcessError(proc.returncode, cmd)
        for names, path in ((SOURCES, LIB_PATH), (PROBE_SOURCES, PROBE_LIB_PATH)):
            objs = [os.path.join(tmp, s.replace(".hip", ".o")) for s in names]
            link = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", path]
            if verbose:
                print(" ".join(link), flush=True)
            subprocess.run(link, check=True)
    return LIB_PATH


if __name__ == "__main__":
    build(extra_flags=sys.argv[1:])
