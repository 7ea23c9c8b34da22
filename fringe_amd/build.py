"""Build libfringe_amd.so in-tree with hipcc for gfx950.

    python -m fringe_amd.build        (or fringe_amd.build.build())

Every HIP translation unit under csrc/ is compiled to an object and linked
into fringe_amd/libfringe_amd.so; the C++ file-level modules (ENVI/VRT I/O,
module processors) are compiled with hipcc too, since they call the HIP
runtime.
"""
import os
import re
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libfringe_amd.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("FRINGE_OFFLOAD_ARCH", "gfx950")

# Packed FP32 instructions are disabled for all device code.
DEVICE_FLAGS = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
# Kernels on the matrix cores may not spill vector registers: a value alike in
# all lanes, spilled under a partial exec mask, has come back without the other
# lanes' share, and pixels with it as zeros.  The compiler's report of these
# sources is read, and the build fails if one does.
RESOURCES = ["-Rpass-analysis=kernel-resource-usage"]
NO_SPILL = ("gram_mfma.hip", "resolve_mfma64.hip", "solve_mfma.hip", "solve_mfma64.hip")
COMMON = ["-O3", "-fPIC", "-std=c++17", f"--offload-arch={ARCH}", "-I" + os.path.join(HERE, "..", "include"),
          "-Wno-unused-result", "-munsafe-fp-atomics"]


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC)
                  if f.endswith(".hip") or f.endswith(".cpp"))


def spilling_kernels(report):
    """[(kernel, vector registers spilled)] of a kernel-resource-usage report,
    and the number of kernels in it."""
    kernels = re.findall(r"Function Name: (\S+)", report)
    spills = [int(k) for k in re.findall(r"VGPRs Spill: (\d+)", report)]
    if len(kernels) != len(spills):
        raise RuntimeError(f"{len(kernels)} kernels but {len(spills)} spill counts in the resource report")
    return [(k, n) for k, n in zip(kernels, spills) if n], len(kernels)


def _compile(src):
    name = os.path.basename(src)
    obj = os.path.join(BUILD, name + ".o")
    guarded = name in NO_SPILL
    cmd = [HIPCC] + (["-x", "hip"] if src.endswith(".cpp") else []) + COMMON + DEVICE_FLAGS
    r = subprocess.run(cmd + (RESOURCES if guarded else []) + ["-c", src, "-o", obj], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stdout}\n{r.stderr}")
    if guarded:
        bad, count = spilling_kernels(r.stderr)
        if bad or not count:
            raise RuntimeError(f"{name}: {count} kernels, vector registers spilled in {bad}")
    return obj


def build(verbose=False):
    os.makedirs(BUILD, exist_ok=True)
    srcs = sources()
    with ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        objs = list(ex.map(_compile, srcs))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp] + objs + ["-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print("built", LIB)
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
