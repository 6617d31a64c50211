"""Build recipe for libinfurnace_hip.so (gfx950 only).

``python -m infurnace_amd.build`` compiles every ``csrc/*.hip`` with hipcc for
gfx950 into ``_build/`` and links ``infurnace_amd/libinfurnace_hip.so`` in
place, beside ``_fast_call.so`` (the wrappers' native argument checks); both are
git-ignored and travel to the GPU box with the source tree.

Packed fp32 VALU forms are switched off for device code
(``-target-feature -packed-fp32-ops``); hipcc's host pass warns that it does
not know the feature, which is harmless.
"""
from __future__ import annotations

import concurrent.futures as cf
import glob
import os
import subprocess
import sys
import sysconfig

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
BUILD_DIR = os.path.join(ROOT, "_build")
LIB_PATH = os.path.join(PKG, "libinfurnace_hip.so")
FAST_PATH = os.path.join(PKG, "_fast_call.so")
ARCH = "gfx950"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
DEVICE_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Wno-unused-function",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


# Per-source extras for the prefill kernels.  They rescale their fp32 accumulators with VALU work
# inside the key loop; with the accumulators in AGPRs the compiler copies all of them to VGPRs and
# back every iteration, so their MFMAs are selected in the VGPR form.  Their maxima run over scores
# that are never NaN for finite inputs (masked keys are -inf), so fmaxf needs no NaN-quieting of
# its operands.  The precondition -- finite queries and K/V -- is part of the documented interface
# (the header's layout notes); with a NaN or Inf among the inputs the prefill output is unspecified.
# The one-launch shared-prefix decode, which runs the prefill body on some of its workgroups, is in
# the same file and shares both.
FILE_FLAGS = {
    "paged_prefill_wide.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form", "-fno-honor-nans"],
    "paged_prefill_block.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form", "-fno-honor-nans"],
    # The whole-row decode kernel's first nine arguments (plan, pool, tables, query, sizes, grid) are
    # preloaded into scalar registers at dispatch, so its first loads (the step plan) do not wait
    # for the kernel-argument loads.
    "paged_decode_rows.hip": ["-mllvm", "-amdgpu-kernarg-preload-count=9"],
}


def _compile(src: str) -> str:
    obj = os.path.join(BUILD_DIR, os.path.basename(src) + ".o")
    extra = FILE_FLAGS.get(os.path.basename(src), [])
    cmd = [HIPCC, *DEVICE_FLAGS, *extra, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    # the only accepted diagnostic noise is the host pass not knowing the gfx feature
    noise = "'-packed-fp32-ops' is not a recognized feature for this target (ignoring feature)"
    err = "\n".join(ln for ln in r.stderr.splitlines() if noise not in ln)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _build_fast() -> str:
    """The wrappers' native argument checks (csrc/fast_call.cpp), a CPython extension against torch's headers."""
    import torch
    troot = os.path.dirname(torch.__file__)
    tmp = FAST_PATH + ".tmp"
    cmd = ["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-isystem", f"{troot}/include",
           "-isystem", sysconfig.get_paths()["include"], "-isystem", "/opt/rocm/include",
           os.path.join(CSRC, "fast_call.cpp"), "-o", tmp, f"-L{troot}/lib", "-lc10", "-lc10_hip", "-ltorch_cpu",
           "-ltorch_python"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed for fast_call.cpp:\n{r.stderr}")
    os.replace(tmp, FAST_PATH)
    return FAST_PATH


def sources() -> list[str]:
    return sorted(glob.glob(os.path.join(CSRC, "*.hip")))


def build(jobs: int = 8) -> str:
    """Compile all HIP sources for gfx950 and link the shared library; returns its path.

    The wrappers' native checks are built beside it where g++ and torch's headers allow; without them the
    wrappers check in Python, so that is a message and no failure."""
    os.makedirs(BUILD_DIR, exist_ok=True)
    srcs = sources()
    with cf.ThreadPoolExecutor(max_workers=max(1, min(jobs, len(srcs)))) as ex:
        fast = ex.submit(_build_fast)
        objs = list(ex.map(_compile, srcs))
    if fast.exception() is not None:
        sys.stderr.write(f"fast_call.cpp is not built, the wrappers' checks run in Python: {fast.exception()}\n")
        if os.path.exists(FAST_PATH):
            os.remove(FAST_PATH)  # (of an earlier build)
    tmp = LIB_PATH + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
    subprocess.run(cmd, check=True)
    # A kernel whose host-side launch stub was not emitted links as an undefined symbol and only fails
    # when the library is loaded; refuse such a library here.
    nm = subprocess.run(["nm", "-u", tmp], capture_output=True, text=True)
    missing = [ln.split()[-1] for ln in nm.stdout.splitlines() if "_ZN3ifn" in ln]
    if missing:
        os.remove(tmp)
        raise RuntimeError(f"{len(missing)} undefined library symbols, e.g. {missing[0]}")
    os.replace(tmp, LIB_PATH)
    return LIB_PATH


if __name__ == "__main__":
    print(build())
