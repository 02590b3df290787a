"""Builds libtbik_hip.so (the gfx950 kernels + their C ABI) in-tree with hipcc, beside it _fast.<python tag>.so (a Python extension
with the common calls of the row-wise operators, host code only) and measure/libtbik_measure.so (the benchmark's machine probes,
which are not part of the product library).

    python -m llm_reproducibility_amd.build            # compile every source, link
    python -m llm_reproducibility_amd.build --if-stale # only when a source is newer than what is built, or torch is another

hipcc cross-compiles for gfx950 without a GPU, so this runs anywhere ROCm is installed.
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
import sysconfig

from . import _lib

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG_DIR, "csrc")
INCLUDE = os.path.join(os.path.dirname(PKG_DIR), "include")
LIB_PATH = os.path.join(PKG_DIR, "libtbik_hip.so")
FAST_SRC = os.path.join(PKG_DIR, "csrc_host", "fast_ops.cpp")
FAST_PATH = os.path.join(PKG_DIR, "_fast" + sysconfig.get_config_var("EXT_SUFFIX"))
MEASURE_DIR = os.path.join(PKG_DIR, "measure")
MEASURE_LIB_PATH = os.path.join(MEASURE_DIR, "libtbik_measure.so")
OBJ_DIR = os.path.join(PKG_DIR, "build")

# -packed-fp32-ops: keep the compiler from forming packed fp32 VALU ops out of scalar float code.
HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-command-line-argument", "-Wno-unknown-warning-option",
]

# Per-file additions.  The hand-ordered GEMM kernels are laid out the way they should issue; the pre-RA machine
# scheduler only lengthens live ranges there (more spills at the 256-register limit), so it is switched off for them.
EXTRA_FLAGS = {
    # Their K loops branch on wave-uniform conditions only (which merge a leaf takes); left unstructured, those branches
    # cost no flow blocks and no register copies at the joins (-structurizecfg-skip-uniform-regions: 252 -> 232 registers
    # and 3 % faster for the first kernel, and what lets the second keep two tree levels in registers without spilling).
    "gemm_tree_wide.hip": ["-mllvm", "-enable-misched=false", "-mllvm", "-structurizecfg-skip-uniform-regions"],
    "gemm_tree_wide_deep.hip": ["-mllvm", "-enable-misched=false", "-mllvm", "-structurizecfg-skip-uniform-regions"],
    # attention rescales its output accumulators every key tile: with the accumulators in ordinary registers that is
    # one multiply each, in accumulation registers it is a read, a multiply and a write back
    "attention.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
}


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def measure_sources():
    return sorted(os.path.join(MEASURE_DIR, f) for f in os.listdir(MEASURE_DIR) if f.endswith(".hip"))


def _deps():
    deps = sources() + measure_sources() + [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".h")]
    deps += [os.path.join(INCLUDE, "tbik_hip.h"), os.path.join(INCLUDE, "tbik_measure.h"), FAST_SRC]
    return deps


def is_stale() -> bool:
    built = (LIB_PATH, MEASURE_LIB_PATH, FAST_PATH)
    if not all(os.path.exists(p) for p in built):
        return True
    with open(FAST_PATH, "rb") as f:
        if _lib.fast_built_for().encode() + b"\0" not in f.read():   # another torch, or another ABI of the library
            return True
    t = min(os.path.getmtime(p) for p in built)
    return any(os.path.getmtime(d) > t for d in _deps())


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found: libtbik_hip.so cannot be built on this machine")
    return exe


def _compile(src: str) -> str:
    obj = os.path.join(OBJ_DIR, os.path.basename(src)[:-4] + ".o")
    cmd = [_hipcc(), *HIPCC_FLAGS, *EXTRA_FLAGS.get(os.path.basename(src), []), "-I", INCLUDE, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{r.stdout}\n{r.stderr}")
    return obj


def _link(objs, path: str) -> None:
    tmp = path + ".tmp"
    cmd = [_hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-fno-gpu-rdc", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, path)


def _compile_fast() -> str:
    import torch
    from torch.utils import cpp_extension

    obj = os.path.join(OBJ_DIR, "fast_ops.o")
    includes = [*cpp_extension.include_paths(), "/opt/rocm/include", sysconfig.get_paths()["include"]]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-Wall", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f'-DTBIK_BUILT_FOR="{_lib.fast_built_for()}"', *[a for p in includes for a in ("-isystem", p)],
           "-c", FAST_SRC, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed on {FAST_SRC}:\n{r.stdout}\n{r.stderr}")
    return obj


def _link_fast(obj: str) -> None:
    import torch

    tmp = FAST_PATH + ".tmp"
    cmd = ["g++", "-shared", "-o", tmp, obj, "-L", os.path.join(os.path.dirname(torch.__file__), "lib"), "-ltorch_cpu", "-ltorch_python",
           "-lc10", "-lc10_hip", "-L", PKG_DIR, "-l:" + os.path.basename(LIB_PATH), "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, FAST_PATH)


def build(verbose: bool = True) -> str:
    os.makedirs(OBJ_DIR, exist_ok=True)
    srcs, msrcs = sources(), measure_sources()
    with cf.ThreadPoolExecutor(max_workers=min(8, len(srcs) + len(msrcs))) as ex:
        fast = ex.submit(_compile_fast)
        objs = list(ex.map(_compile, srcs + msrcs))
        fast_obj = fast.result()
    _link(objs[:len(srcs)], LIB_PATH)
    _link(objs[len(srcs):], MEASURE_LIB_PATH)
    _link_fast(fast_obj)
    if verbose:
        print(f"built {LIB_PATH} from {len(srcs)} sources and {MEASURE_LIB_PATH} from {len(msrcs)}")
    return LIB_PATH


def main(argv=None) -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--if-stale", action="store_true")
    args = ap.parse_args(argv)
    if args.if_stale and not is_stale():
        print(f"{LIB_PATH} is up to date")
        return 0
    build()
    return 0


if __name__ == "__main__":
    sys.exit(main())
