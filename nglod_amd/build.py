"""Builds libnglod_hip.so (gfx950) in-tree with hipcc.

Usage: python -m nglod_amd.build   (or nglod_amd.build.build_library()).
"""
import os
import subprocess
import sys
import concurrent.futures as cf

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "libnglod_hip.so")
OBJDIR = os.path.join(HERE, "_build")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
]


# Per-file additions.  mixed.hip (the mixed-form trace passes): MFMA results
# in ordinary VGPRs.  Those kernels read every output element with the vector
# ALU (ReLU, second layer); the AGPR form costs a v_accvgpr_read per element
# and the AGPRs themselves (pass 1: 134 VGPRs instead of 152 + 16 AGPRs, 3-4%
# faster on the 1280x720 frame; the batch-query kernels measured slower with
# it and keep the default).
EXTRA = {
    "mixed.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
    "sol_march.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
    "trace_group.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
    "query_cells.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
}


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def _compile(src):
    obj = os.path.join(OBJDIR, os.path.basename(src) + ".o")
    cmd = [HIPCC, *FLAGS, *EXTRA.get(os.path.basename(src), []), "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stdout}\n{r.stderr}")
    return obj


def build_library(verbose=True):
    os.makedirs(OBJDIR, exist_ok=True)
    srcs = sources()
    with cf.ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        objs = list(ex.map(_compile, srcs))
    tmp = OUT + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, OUT)
    if verbose:
        print(f"built {OUT}")
    return OUT


if __name__ == "__main__":
    build_library()
    sys.exit(0)
