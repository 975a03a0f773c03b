"""Build libstile_hip.so in-tree for gfx950 with hipcc.

The library is a plain C-ABI shared object (include/stile.h); Python reaches
it through ctypes (stile_amd/_native.py).  It is built in place, next to its
sources, so the built file travels with the source tree.
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_DIR = os.path.join(HERE, "_lib")
LIB_PATH = os.path.join(LIB_DIR, "libstile_hip.so")
SOURCES = ["stile_kernels.hip", "stile_attention.hip", "stile_sparse.hip",
           "stile_stream.hip", "stile_dense.hip", "stile_sddmm.hip",
           "stile_plan.hip"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

# -packed-fp32-ops off: hipcc -O3 otherwise forms v_pk_{add,mul,fma}_f32 from
# scalar and float2 code on its own.
COMMON_FLAGS = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-result",
]


def build_native(verbose=False):
    """Compile every HIP source and link libstile_hip.so (always rebuilds)."""
    os.makedirs(LIB_DIR, exist_ok=True)
    objs = [os.path.join(LIB_DIR, os.path.splitext(src)[0] + ".o") for src in SOURCES]
    cmds = [[HIPCC, *COMMON_FLAGS, "-c", os.path.join(CSRC, src), "-o", obj] for src, obj in zip(SOURCES, objs)]
    with ThreadPoolExecutor(4) as pool:   # the sources compile side by side
        list(pool.map(lambda cmd: _run(cmd, verbose), cmds))
    tmp = LIB_PATH + ".tmp"
    _run([HIPCC, "-shared", f"--offload-arch={ARCH}", "-fPIC", *objs, "-o", tmp], verbose)
    os.replace(tmp, LIB_PATH)
    for o in objs:
        os.remove(o)
    return LIB_PATH


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in r.stdout.splitlines()
                    if "packed-fp32-ops' is not a recognized feature" not in l)
    if verbose and out.strip():
        print(out)
    if r.returncode != 0:
        raise RuntimeError(f"build failed ({r.returncode}): {' '.join(cmd)}\n{out}")


if __name__ == "__main__":
    print(build_native(verbose="-v" in sys.argv))
