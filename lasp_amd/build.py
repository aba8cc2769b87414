"""Builds lasp_amd/liblasp_hip.so for gfx950 with hipcc (cross-compiles without a GPU).

    python -m lasp_amd.build
"""
import os
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "liblasp_hip.so")
SOURCES = ["lasp_abi.hip", "lasp_generic.hip", "lasp_mfma.hip", "lasp_mfma_f16.hip", "lasp_mfma_f32.hip", "lasp_probe.hip"]

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
    return LIB


if __name__ == "__main__":
    build(extra_flags=sys.argv[1:])
