"""Builds libmumfim_amd.so (host C++ + HIP kernels for gfx950) in-tree.

Each source compiles to an object under mumfim_amd/_build/ and the objects
link into mumfim_amd/libmumfim_amd.so.  FP64 kernel files are compiled with
-ffp-contract=off so their arithmetic rounds like the reference C++.
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libmumfim_amd.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

COMMON = ["-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function"]
DEVICE = [f"--offload-arch={ARCH}",
          # packed FP32 math stays off on this hardware
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
SOURCES = {
    "network.cpp": [],
    "api.cpp": [],
    "fe2.cpp": [],
    "aux_kernels.hip": ["-ffp-contract=off"],
    # constants of the exponential stay where they are used: moved out of the
    # step loop they take some 30 registers a lane, which then spill
    "solve64.hip": ["-ffp-contract=off", "-mllvm", "-disable-machine-licm"],
    "solve64l.hip": ["-ffp-contract=off"],
    "solve32.hip": [],
    "solve32t.hip": [],
    # values stay where they are used: moved out of the step loop they spill
    "solve32tk.hip": ["-mllvm", "-disable-machine-licm"],
    "mlp.hip": [],
}


def _compile(src, extra):
    obj = os.path.join(BUILD, src + ".o")
    lang = ["-x", "hip"] if src.endswith(".cpp") else []
    cmd = [HIPCC, "-c"] + lang + [os.path.join(CSRC, src), "-o", obj] + COMMON + DEVICE + extra
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"compile failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    if r.stderr.strip():
        warn = [l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l and l.strip()]
        if warn:
            sys.stderr.write("\n".join(warn) + "\n")
    return obj


def build(verbose=True):
    os.makedirs(BUILD, exist_ok=True)
    jobs = min(len(SOURCES), os.cpu_count() or 4)
    with ThreadPoolExecutor(jobs) as ex:
        objs = list(ex.map(lambda kv: _compile(*kv), SOURCES.items()))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "-shared", "-o", tmp] + objs + [f"--offload-arch={ARCH}", "-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build()
