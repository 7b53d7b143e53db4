"""Builds the HIP library in-tree: resolve2d_amd/lib/libr2d_hip.so (gfx950).

Flags: -ffp-contract=off keeps every f32 expression a separate IEEE operation
(the reference's strict float mode); f32 division and sqrt stay correctly
rounded (HIP's default); packed-fp32 instruction selection is disabled.  The
VGPR live-range pass is off: with it the compiler's own machine verifier
(-mllvm -verify-machineinstrs) refuses the larger device functions here, and
without it they all pass (same speed).
"""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIBDIR, "libr2d_hip.so")
SOURCES = ["r2d_kernels.hip", "r2d_api.hip"]
HEADERS = ["r2d_math.h", "r2d_device.h", "r2d_chain.h", "r2d_kernels.h", os.path.join("..", "..", "include", "r2d.h")]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("R2D_OFFLOAD_ARCH", "gfx950")
FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
    "-fvisibility=hidden", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result", "-Xarch_device", "-mllvm=-amdgpu-opt-vgpr-liverange=0",
    # loops of one wave start at a cache line (20-row pyramid step 261 -> 256 us, 1,024 worlds 27.7 -> 27.3 ms)
    "-Xarch_device", "-mllvm=-align-all-nofallthru-blocks=6",
]


def verify(out_dir: str) -> list:
    """Compile every source with the compiler's machine verifier on (a minute
    and a half, so not part of build) and return what it refused: (source,
    messages).  A kernel that outgrew its registers has come out of the
    compiler with an undefined register, and faulted."""
    runs = []
    for src in SOURCES:
        cmd = [HIPCC] + FLAGS + ["-Xarch_device", "-mllvm=-verify-machineinstrs", "-c", os.path.join(CSRC, src), "-o",
                                 os.path.join(out_dir, src + ".o")]
        runs.append((src, subprocess.Popen(cmd, stdout=subprocess.DEVNULL, stderr=subprocess.PIPE, text=True)))
    done = [(src, p.communicate()[1], p.returncode) for src, p in runs]
    return [(src, err) for src, err, rc in done if rc != 0]


def build(verbose: bool = False) -> str:
    os.makedirs(LIBDIR, exist_ok=True)
    objs = []
    for src in SOURCES:
        obj = os.path.join(LIBDIR, src.replace(".hip", ".o"))
        cmd = [HIPCC] + FLAGS + ["-c", os.path.join(CSRC, src), "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.run(cmd, check=True, stderr=None if verbose else subprocess.DEVNULL)
        objs.append(obj)
    tmp = LIB + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp] + objs
    subprocess.run(cmd, check=True)
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
