"""Builds the gfx950 kernel library in-tree with hipcc.

    python -m logismos_amd.build

produces ``logismos_amd/lib/liblogismos_kernels.so`` (the C-ABI declared in
``include/logismos_decode.h``) and ``liblogismos_kernels.a`` (the static
archive a Rust `kernels` build script would link, mirroring
crates/kernels/build.rs:71-124 of the reference with
``--offload-arch=gfx950`` and wave64).
"""
from __future__ import annotations

import glob
import os
import re
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
OBJDIR = os.path.join(LIBDIR, "obj")
SO_PATH = os.path.join(LIBDIR, "liblogismos_kernels.so")
A_PATH = os.path.join(LIBDIR, "liblogismos_kernels.a")

OFFLOAD_ARCH = os.environ.get("LOGISMOS_OFFLOAD_ARCH", "gfx950")

# -packed-fp32-ops is switched off: the compiler must not form v_pk_*_f32.
# The first 16 dwords of a kernel's scalar arguments arrive in scalar registers with the wave
# instead of being loaded by it: about 0.2 us of every small launch (a 36-layer step of 32 rows
# 5.61 -> 5.52 ms, one 12288 x 4096 product of 8 rows 8.50 -> 8.25 us).
HIPCC_FLAGS = [
    f"--offload-arch={OFFLOAD_ARCH}", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=fast",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
    "-Wall", "-Wno-unused-function", "-Wno-unknown-attributes",
]


# Per-source additions.  paged_attn.hip: MFMA results stay in ordinary VGPRs (the
# kernels fit in 256 registers; the default accumulation-register form costs the
# prefill kernel ~50 register-to-register moves per key tile around its softmax).
EXTRA_FLAGS = {
    "paged_attn.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
    "qgemm_q4_splitk.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
    "qgemm_q4_stream.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
    "qgemm_q4_greedy.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
    "decode_resident.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
    "qgemm_q4_rows.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
    "ref_ops.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
    "paged_attn_chunk64.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
    "qgemm_q4g32.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
}

# Kernels that ask for operands in one assembly statement and wait for them in a later one, so that
# work lies between the two.  A register that the compiler moved to memory (or copied) in between
# would keep what it held before the read, with no error: a build in which one of them spills is refused.  So is one of
# decode_resident_kernel, whose requests go straight into LDS: there a reload from scratch waits for all of them
# (24 layers of width 896 6 % slower).
READS_IN_FLIGHT = ("qgemm_q4g128_tallp_kernel", "matmul_ring_fp16_kernel", "paged_attn_chunk64_kernel",
                   "decode_resident_kernel")


def spills(remarks: str) -> list[str]:
    """The kernels of READS_IN_FLIGHT that use scratch memory, from the compiler's
    kernel-resource-usage remarks."""
    found, name = [], ""
    for line in remarks.splitlines():
        if m := re.search(r"remark: Function Name: (\S+)", line):
            name = m.group(1)
        elif m := re.search(r"remark:\s+(VGPRs Spill|ScratchSize \[bytes/lane\]): ([1-9]\d*)", line):
            if any(k in name for k in READS_IN_FLIGHT):
                found.append(f"{name}: {m.group(1)} {m.group(2)}")
    return found


def hipcc() -> str:
    exe = os.environ.get("HIPCC") or shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe) and not shutil.which(exe):
        raise RuntimeError("hipcc not found (set HIPCC); the kernels cannot be built")
    return exe


def sources() -> list[str]:
    return sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.cpp")))


def _compile(src: str) -> str:
    obj = os.path.join(OBJDIR, os.path.basename(src) + ".o")
    cmd = [hipcc(), *HIPCC_FLAGS, *EXTRA_FLAGS.get(os.path.basename(src), []),
           "-Rpass-analysis=kernel-resource-usage", "-fno-caret-diagnostics", "-x", "hip", "-c", src,
           "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr}")
    if bad := spills(r.stderr):
        os.remove(obj)
        raise RuntimeError(f"{src}: registers spilled where reads are in flight:\n" + "\n".join(bad))
    noise = ("packed-fp32-ops", "is not a recognized feature", "[-Rpass-analysis=")
    warn = [ln for ln in r.stderr.splitlines() if ln.strip() and not any(n in ln for n in noise)]
    if warn:
        sys.stderr.write("\n".join(warn) + "\n")
    return obj


def build(verbose: bool = True) -> str:
    os.makedirs(OBJDIR, exist_ok=True)
    srcs = sources()
    with ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        objs = list(ex.map(_compile, srcs))
    r = subprocess.run([hipcc(), f"--offload-arch={OFFLOAD_ARCH}", "-shared", "-fPIC", "-o",
                        SO_PATH, *objs], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    if os.path.exists(A_PATH):
        os.remove(A_PATH)
    subprocess.run(["ar", "crs", A_PATH, *objs], check=True)
    if verbose:
        print(f"built {SO_PATH} from {len(srcs)} sources for {OFFLOAD_ARCH}")
    return SO_PATH


if __name__ == "__main__":
    build()
