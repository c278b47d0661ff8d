"""Builds libzenyx_kv.so in-tree from zenyx_amd/csrc/*.hip for gfx950 with hipcc.

Every translation unit is compiled to its own object (in parallel), then linked into
zenyx_amd/lib/libzenyx_kv.so, which is written atomically so a concurrent loader never
sees a half-written file.
"""
from __future__ import annotations

import concurrent.futures as cf
import glob
import os
import shutil
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_DIR = os.path.join(HERE, "lib")
OBJ_DIR = os.path.join(LIB_DIR, "_build")
LIB = os.path.join(LIB_DIR, "libzenyx_kv.so")

ARCH = "gfx950"
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    # exact IEEE arithmetic: the kernels are compared bit-for-bit with a CPU oracle
    "-ffp-contract=off", "-fno-fast-math",
    # torch's bundled HIP runtime loads these code objects
    "-mcode-object-version=5",
    # no packed fp32 ops (v_pk_*_f32) anywhere in this library
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]
# per-file options:
# * append: under this machine scheduler the fused append's loads issue in longer clauses
#   (0.5-0.8% less time per 32-layer x 74,902-token append on MI355X, same codes);
# * prefill: matrix results in vector registers.  By default a kernel that may use more than
#   256 registers takes them in accumulation registers, and the 64-row kernel copied every
#   score out again (64 moves per step, and spills).
FILE_FLAGS = {"zx_append_fused.hip": ["-mllvm", "-amdgpu-sched-strategy=max-memory-clause"],
              "zx_prefill.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"]}


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(path):
        raise RuntimeError("hipcc not found (ROCm is required to build libzenyx_kv.so)")
    return path


def _compile(src: str) -> str:
    obj = os.path.join(OBJ_DIR, os.path.basename(src) + ".o")
    cmd = [hipcc(), *HIPCC_FLAGS, *FILE_FLAGS.get(os.path.basename(src), []), "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{r.stdout}\n{r.stderr}")
    return obj


def build(verbose: bool = False) -> str:
    """Compile every csrc/*.hip and link libzenyx_kv.so (returns its path)."""
    os.makedirs(OBJ_DIR, exist_ok=True)
    sources = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    if not sources:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    workers = min(len(sources), max(1, (os.cpu_count() or 4) // 2), 8)
    with cf.ThreadPoolExecutor(workers) as ex:
        objs = list(ex.map(_compile, sources))
    tmp = LIB + f".tmp{os.getpid()}"
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link of libzenyx_kv.so failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB} from {len(sources)} sources")
    return LIB


if __name__ == "__main__":
    build(verbose=True)
