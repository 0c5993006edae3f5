"""Builds ``liblattice_hip_q4.so`` for gfx950 with hipcc, and ``_lq4_py.so`` (its CPython entry), in-tree, next to this
file.

``python -m lattice_amd.build`` compiles every translation unit under ``csrc/``
(in parallel) and links them.  hipcc cross-compiles, so no GPU is needed to build.
"""
from __future__ import annotations

import os
import shlex
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "liblattice_hip_q4.so")
PY_EXT = os.path.join(HERE, "_lq4_py.so")
SOURCES = ["lq4_api.hip", "lq4_gemv.hip", "lq4_gemv_b1.hip", "lq4_gemv_dma.hip", "lq4_gemv_multi.hip", "lq4_gemv_i8.hip", "lq4_gemv_mfma.hip", "lq4_gemm.hip", "lq4_gemm_wreg.hip", "lq4_gemm_skinny.hip", "lq4_moe.hip", "lq4_moe_i8.hip", "lq4_moe_gemm.hip", "lq4_moe_b1.hip", "lq4_topk.hip", "lq4_elementwise.hip", "lq4_q8.hip", "lq4_q3.hip"]

# -packed-fp32-ops: keep the compiler from forming v_pk_*_f32 out of scalar float code.
# kernarg preload: the first sixteen dwords of a kernel's arguments arrive in scalar registers with the wave instead of
# through a scalar load at its start, which the first memory request of a launch would wait for (six 26.7 MB Q8_0 GEMVs
# 50.5 -> 48.0 us, an eight-row decode layer 42.1 -> 41.1).
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-mllvm", "-amdgpu-kernarg-preload-count=16"]
_NOISE = "'-packed-fp32-ops' is not a recognized feature for this target"  # host pass only


def _run(cmd):
    p = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in p.stderr.splitlines() if _NOISE not in l)
    if p.returncode != 0:
        raise RuntimeError(f"command failed: {' '.join(cmd)}\n{p.stdout}\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")


def build(verbose: bool = False) -> str:
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    extra = shlex.split(os.environ.get("LQ4_CXXFLAGS", ""))  # e.g. -DNAME for experiments
    objs = [os.path.join(CSRC, s.replace(".hip", ".o")) for s in SOURCES]

    def compile_one(pair):
        src, obj = pair
        cmd = [hipcc, *FLAGS, *extra, "-c", os.path.join(CSRC, src), "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        _run(cmd)

    with ThreadPoolExecutor(max_workers=min(4, len(SOURCES))) as ex:
        list(ex.map(compile_one, zip(SOURCES, objs)))
    _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB, *objs])
    # the CPython entry: host code only, resolves the library next to itself
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall",
           "-I" + sysconfig.get_paths()["include"], os.path.join(CSRC, "lq4_py.cpp"), "-o", PY_EXT, "-L" + HERE,
           "-l:" + os.path.basename(LIB), "-Wl,-rpath,$ORIGIN"]
    if verbose:
        print(" ".join(cmd), flush=True)
    _run(cmd)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
