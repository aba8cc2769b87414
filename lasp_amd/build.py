"""Builds lasp_amd/liblasp_hip.so for gfx950 with hipcc (cross-compiles without a GPU) and lasp_amd/_lasp_torch.so.

    python -m lasp_amd.build
"""
import os
import subprocess
import sys
import sysconfig
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "liblasp_hip.so")
TORCH_LIB = os.path.join(HERE, "_lasp_torch.so")
SOURCES = ["lasp_abi.hip", "lasp_generic.hip", "lasp_mfma.hip", "lasp_mfma_f16.hip", "lasp_mfma_f32.hip", "lasp_probe.hip", "lasp_step.hip"]

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    "-I", os.path.join(ROOT, "include"),
    "-I", CSRC,
]


def build(verbose: bool = True, extra_flags=()) -> str:
    """Compiles every source to an object of its own, side by side, and links them."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    compile_flags = [f for f in HIPCC_FLAGS if f != "-shared"]
    with tempfile.TemporaryDirectory() as tmp:
        objects = [os.path.join(tmp, s + ".o") for s in SOURCES]

        def compile_one(job):
            src, obj = job
            cmd = [hipcc, *compile_flags, *extra_flags, "-c", os.path.join(CSRC, src), "-o", obj]
            if verbose:
                print(" ".join(cmd), flush=True)
            subprocess.run(cmd, check=True)

        with ThreadPoolExecutor(max_workers=min(len(SOURCES), os.cpu_count() or 1)) as pool:
            list(pool.map(compile_one, zip(SOURCES, objects)))
        cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *objects, "-o", LIB]
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.run(cmd, check=True)
    build_torch_side(verbose)
    return LIB


def build_torch_side(verbose: bool = True) -> str:
    """Compiles lasp_torch.cpp, host code over the library's C ABI, against torch's headers."""
    import torch

    base = os.path.dirname(os.path.abspath(torch.__file__))
    include = [os.path.join(base, "include"), os.path.join(base, "include", "torch", "csrc", "api", "include"),
               os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"), sysconfig.get_paths()["include"],
               os.path.join(ROOT, "include")]
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *[x for path in include for x in ("-isystem", path)], os.path.join(CSRC, "lasp_torch.cpp"), "-o", TORCH_LIB,
           "-L" + HERE, "-llasp_hip", "-L" + os.path.join(base, "lib"), "-ltorch_python", "-ltorch_cpu", "-ltorch", "-lc10",
           "-lc10_hip", "-Wl,-rpath,$ORIGIN"]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    return TORCH_LIB


if __name__ == "__main__":
    build(extra_flags=sys.argv[1:])
