"""Build recipe for libexl3moe.so (gfx950) -- run by __graft_entry__.build().

Every HIP translation unit under exl3-server_amd/csrc is compiled with hipcc for gfx950
(in parallel), then linked into exl3-server_amd/exl3_amd/libexl3moe.so, in-tree so it
travels with the repository snapshot.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import subprocess
import sys

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG_DIR)                # exl3-server_amd/
REPO = os.path.dirname(ROOT)
CSRC = os.path.join(ROOT, "csrc")
INCLUDE = os.path.join(REPO, "include")
BUILD_DIR = os.path.join(ROOT, "_build")
LIB_PATH = os.path.join(PKG_DIR, "libexl3moe.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

# -ffp-contract=off: every multiply/add the kernels spell separately stays separately
# rounded (the bit-exact reconstruct and Hadamard steps depend on it); fused operations
# are requested explicitly (fmaf, v_dot2, v_pk_fma_f16).
# The packed-fp32 feature is switched off for the device code: the hardware packed f32
# ops are kept out of every kernel.
CFLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
    f"-I{INCLUDE}", f"-I{CSRC}",
]

# the expert kernels' instantiations are spread over moe_experts_k*.hip so that they compile
# in parallel (the longest first)
SOURCES = ["moe_experts_k78.hip", "moe_experts_k56.hip", "moe_experts_k34.hip", "moe_experts_k12.hip",
           "qmv_rows_k58.hip", "qmv_rows_k14.hip",
           "trellis_kernels.hip", "moe_experts.hip", "moe_shared.hip", "moe.hip", "api.hip", "loader.hip", "hc.hip"]


def _compile(src: str) -> str:
    obj = os.path.join(BUILD_DIR, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC, *CFLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in (r.stderr or "").splitlines() if noise not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{err}")
    if err.strip():
        print(err, file=sys.stderr)
    return obj


def build(jobs: int | None = None) -> str:
    os.makedirs(BUILD_DIR, exist_ok=True)
    jobs = jobs or min(len(SOURCES), os.cpu_count() or 1)
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(_compile, SOURCES))
    tmp = LIB_PATH + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    os.replace(tmp, LIB_PATH)
    return LIB_PATH


if __name__ == "__main__":
    print(build())
