"""Ahead-of-time build of libhtr_gfx950.so with hipcc (gfx950 only).

The reference JIT-builds its extension on first use (htr/ops.py:11-21 of the reference); here the
library is compiled explicitly and kept in-tree next to its source, and importing the package never
compiles anything.  Run `python -m htr_amd.build`.
"""
import os
import subprocess
import sys

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "csrc")
LIB = os.path.join(CSRC, "libhtr_gfx950.so")
SOURCES = [os.path.join(CSRC, "htr_gfx950.hip")]          # one translation unit; the kernels live in the parts it includes
PARTS = [os.path.join(CSRC, f) for f in ("decode.hpp", "linear.hpp", "linear_batch.hpp", "linear_tile.hpp", "linear_gemm.hpp", "linear_wide.hpp", "moe.hpp", "dequant.hpp",
                                         "viterbi.hpp", "anchors.hpp", "plan.hpp")]
BINDING_SOURCE = os.path.join(CSRC, "torch_binding.cpp")
BINDING = os.path.join(os.path.dirname(CSRC), "_fast.so")
HEADER = os.path.join(os.path.dirname(CSRC), os.pardir, "include", "htr_gfx950.h")

HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-shared", "-fPIC",
    # keep the compiler from forming packed-FP32 VALU instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]


def hipcc():
    return os.environ.get("HIPCC") or os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")


def binding_command():
    """The host-only extension htr_amd._fast: torch's headers, g++; no kernel in it."""
    import sysconfig
    import torch
    root = os.path.dirname(torch.__file__)
    lib = os.path.join(root, "lib")
    return [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-shared", "-fPIC", "-Wall",
            f'-DHTR_BUILD_TORCH="{torch.__version__}"', f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
            "-I" + os.path.join(root, "include"), "-I" + os.path.join(root, "include", "torch", "csrc", "api", "include"),
            "-I" + sysconfig.get_paths()["include"], BINDING_SOURCE, "-o", BINDING, "-L" + lib, "-lc10", "-ltorch_cpu", "-ltorch_python"]


def build(verbose=False, extra=()):
    cmds = [[hipcc()] + HIPCC_FLAGS + list(extra) + ["-o", LIB] + SOURCES, binding_command()]
    if verbose:
        for cmd in cmds:
            print(" ".join(cmd), flush=True)
    procs = [subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True) for cmd in cmds]
    outs = [p.communicate()[0] for p in procs]
    for cmd, p, text in zip(cmds, procs, outs):
        out = "\n".join(l for l in text.splitlines() if "not a recognized feature" not in l)
        if p.returncode != 0:
            raise RuntimeError(os.path.basename(cmd[0]) + " failed:\n" + out)
        if verbose and out.strip():
            print(out)
    return LIB


def is_stale():
    def older(built, sources):
        return not os.path.exists(built) or any(os.path.getmtime(s) > os.path.getmtime(built) for s in sources)
    return older(LIB, SOURCES + PARTS + [HEADER]) or older(BINDING, [BINDING_SOURCE, HEADER])


if __name__ == "__main__":
    print(build(verbose=True, extra=sys.argv[1:]))
