"""Build recipe of librome_gpu.so (hipcc, gfx950), in-tree next to this file.

    python -m rome_amd.build          # compile every source, link rome_amd/librome_gpu.so
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "librome_gpu.so")
OBJ = os.path.join(HERE, "_build")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

SOURCES = ["kernels.hip", "gemm_lowp.hip", "weights.hip", "backproject.hip", "fourier_map.hip", "reconstruct.hip", "gridding.hip", "imageprep.hip",
           "proposal.hip", "noalloc.hip",
           "engine.cpp", "sampling.cpp", "mstep.cpp"]
FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-munsafe-fp-atomics",
    # packed FP32 VALU ops are kept off on this target
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # host arithmetic must not contract (pose tables are compared bit for bit)
    "-Xarch_host", "-ffp-contract=off",
    "-Wall", "-Wno-unused-function",
]
# vectors of equal scalars (8 registers each) made ahead of k_gemm_pq_cols' loop spilled 1.5 KB a lane
FILE_FLAGS = {"gemm_lowp.hip": ["-fno-slp-vectorize"]}


def _compile(src):
    obj = os.path.join(OBJ, src + ".o")
    cmd = [HIPCC] + FLAGS + FILE_FLAGS.get(src, []) + ["-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{err}")
    return obj


def build(verbose=False):
    os.makedirs(OBJ, exist_ok=True)
    with ThreadPoolExecutor(max_workers=len(SOURCES)) as ex:
        objs = list(ex.map(_compile, SOURCES))
    tmp = OUT + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp] + objs + [
        "-L/opt/rocm/lib", "-lhipfft", "-Wl,-rpath,/opt/rocm/lib"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stderr)
    os.replace(tmp, OUT)
    if verbose:
        print("built", OUT)
    return OUT


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
