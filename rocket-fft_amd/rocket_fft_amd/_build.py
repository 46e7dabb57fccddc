"""Builds the gfx950 shared library librocketfft_hip.so in place.

hipcc compiles each HIP source of ``rocket-fft_amd/csrc`` to an object in
``rocket-fft_amd/_build`` (in parallel), then links the shared library next
to this file.  Packed FP32 instructions are disabled for all device code.
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
PKG_ROOT = os.path.dirname(HERE)
CSRC = os.path.join(PKG_ROOT, "csrc")
BUILD = os.path.join(PKG_ROOT, "_build")
LIB = os.path.join(HERE, "librocketfft_hip.so")
SOURCES = ["fast.hip", "fast64.hip", "lines_c2c.hip", "lines_blue.hip", "lines_real.hip", "lines_r2r.hip",
           "ragged.hip", "plan.hip", "kernels.hip", "mfma.hip", "pass1024.hip", "pipe4096.hip",
           "engine.hip", "lineops.hip"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "-O3", "-std=c++17", "--offload-arch=gfx950", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]
# The general line kernel holds every radix in one loop over the stages;
# hoisting their constants and strides out of it costs hundreds of spilled
# scalar registers.
FILE_FLAGS = {s: ["-mllvm", "-disable-machine-licm"]
              for s in ("lines_c2c.hip", "lines_blue.hip", "lines_real.hip", "lines_r2r.hip",
                        "ragged.hip")}


def _compile(src):
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC, *FLAGS, *FILE_FLAGS.get(src, []), "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr}")
    return obj


def build(verbose=True):
    os.makedirs(BUILD, exist_ok=True)
    with ThreadPoolExecutor(max_workers=len(SOURCES)) as ex:
        objs = list(ex.map(_compile, SOURCES))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "-shared", "--offload-arch=gfx950", "-fPIC", *objs, "-o", tmp]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}", file=sys.stderr)
    return LIB


if __name__ == "__main__":
    build()
