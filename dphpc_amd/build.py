"""Compile the HIP library for gfx950 with hipcc (cross-compiles without a GPU)."""
import os
import shutil
import subprocess
import tempfile

PKG = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG, "csrc")
LIB_DIR = os.path.join(PKG, "lib")
LIB_PATH = os.path.join(LIB_DIR, "libsddmm_amd.so")

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",          # FMAs are written explicitly; the exact kernel needs mul and add apart
    "-fno-gpu-rdc",
    "-Wall",
    "-Wno-unused-function",
    # packed fp32 VALU forms are kept out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # the first 14 words of a kernel's arguments are in registers when it starts: a wavefront of a short launch has one or
    # two dependent loads less before its first gather (dense tiles K = 512 bf16 16.5 -> 16.1 us, short launches 2 .. 7 %)
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
]


def hipcc():
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found")


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def build_library(verbose=False, extra_flags=(), out=None):
    """(Re)build dphpc_amd/lib/libsddmm_amd.so; returns its path.  The translation units are compiled side by side."""
    os.makedirs(LIB_DIR, exist_ok=True)
    out = out or LIB_PATH
    with tempfile.TemporaryDirectory() as tmp:
        jobs, objects = [], []
        for src in sources():
            obj = os.path.join(tmp, os.path.basename(src) + ".o")
            cmd = [hipcc()] + HIPCC_FLAGS + list(extra_flags) + ["-c", "-o", obj, src]
            if verbose:
                print(" ".join(cmd), flush=True)
            jobs.append((cmd, subprocess.Popen(cmd)))
            objects.append(obj)
        failed = [cmd for cmd, job in jobs if job.wait() != 0]
        if failed:
            raise subprocess.CalledProcessError(1, failed[0])
        subprocess.check_call([hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", out] + objects)
    return out


if __name__ == "__main__":
    print(build_library(verbose=True))
