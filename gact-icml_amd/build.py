"""Build libgact_hip.so (the C-ABI library of HIP kernels) and libgact_probe.so (compute-free traffic probes that
bench.py measures beside the kernels) for gfx950 with hipcc, and gact_torch.so (the operators' host side on torch tensors,
which calls libgact_hip.so) with the host compiler.

    python gact-icml_amd/build.py            # build if the sources are newer than the library
    python gact-icml_amd/build.py --force

hipcc cross-compiles for gfx950 without a GPU present.  The library lands inside the Python
package (gact/lib/) so that it travels with the source tree.
"""
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
SRC = os.path.join(HERE, "csrc", "gact_hip.hip")
PROBE_SRC = os.path.join(HERE, "csrc", "stream_probe.hip")   # compute-free traffic probes for bench.py
HDR = os.path.join(ROOT, "include", "gact_hip.h")
OUT_DIR = os.path.join(HERE, "gact", "lib")
OUT = os.path.join(OUT_DIR, "libgact_hip.so")
TORCH_SRC = os.path.join(HERE, "csrc", "torch_ops.cpp")
TORCH_OUT = os.path.join(OUT_DIR, "gact_torch.so")
PROBE_OUT = os.path.join(OUT_DIR, "libgact_probe.so")

HIPCC_FLAGS = [
    "-O3",
    "--offload-arch=gfx950",
    "-std=c++17",
    "-fPIC",
    "-shared",
    # every floating-point operation in the kernels is meant literally (the one FMA is spelled out)
    "-ffp-contract=off",
    # keep the compiler from forming packed-FP32 instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # the first 16 dwords of a kernel's arguments arrive in scalar registers with the wave (gfx950 preloads them) instead
    # of through a load that every wave waits for before it can ask for data: dequantize of a 16 MB float tensor
    # 4.40 -> 4.22 us, of a 34 MB half tensor 9.15 -> 9.02, large tensors 0.5-1 %.  The quantize kernels, which lose up
    # to 0.5 % by it, take a structure as their first argument and so stay as they were.
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
    "-Wall",
    "-Wno-unused-command-line-argument",
]


def hipcc():
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (set HIPCC)")


def up_to_date():
    built = (OUT, PROBE_OUT, TORCH_OUT)
    if not all(os.path.exists(p) for p in built):
        return False
    with open(TORCH_OUT, "rb") as f:
        if torch_mark() not in f.read():     # built for another torch
            return False
    t = min(os.path.getmtime(p) for p in built)
    return all(os.path.getmtime(p) <= t for p in (SRC, PROBE_SRC, TORCH_SRC, HDR, os.path.abspath(__file__)))


def torch_mark():
    """What gact_torch.so holds of the torch whose headers and libraries it was built with (gact_torch.torch_version)."""
    import torch

    return b"torch " + torch.__version__.encode() + b"\0"


def torch_command():
    """The host compiler's line for gact_torch.so: torch's headers and libraries, ROCm's headers, Python's headers."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    libs = os.path.join(os.path.dirname(torch.__file__), "lib")
    cmd = [os.environ.get("CXX") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           "-D_GLIBCXX_USE_CXX11_ABI=%d" % int(torch._C._GLIBCXX_USE_CXX11_ABI),
           '-DGACT_TORCH_VERSION="%s"' % torch.__version__, "-I", os.path.join(ROOT, "include")]
    for path in cpp_extension.include_paths("cuda") + [sysconfig.get_paths()["include"]]:
        cmd += ["-isystem", path]
    # libtorch.so itself stays out: it would pull in every library torch was built with
    return cmd + ["-o", TORCH_OUT, TORCH_SRC, "-L", OUT_DIR, "-l:libgact_hip.so", "-L", libs, "-ltorch_python", "-ltorch_cpu", "-lc10",
                  "-lc10_hip", "-Wl,-rpath,$ORIGIN"]


def build(force=False, extra=()):
    if not force and up_to_date():
        return OUT
    os.makedirs(OUT_DIR, exist_ok=True)
    cmd = [hipcc()] + HIPCC_FLAGS + list(extra) + ["-I", os.path.join(ROOT, "include"), "-o", OUT, SRC]
    subprocess.run(cmd, check=True)
    subprocess.run([hipcc()] + HIPCC_FLAGS + ["-o", PROBE_OUT, PROBE_SRC], check=True)
    subprocess.run(torch_command(), check=True)
    return OUT


if __name__ == "__main__":
    print(build(force="--force" in sys.argv))
