"""Builds liboctofmm.so (gfx950) in-tree with hipcc.

    python -m octotiger_amd.build          # library
    python -m octotiger_amd.build --asm    # also dump the gfx950 assembly to _build/
"""
import hashlib
import os
import re
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "liboctofmm.so")
SOURCES = ["octofmm.hip", "stencil.cpp"]
HEADERS = ["kernels.hpp", "octofmm_internal.hpp"]
ARCH = os.environ.get("OCTOFMM_ARCH", "gfx950")

# Packed FP32 instructions stay disabled for every device compile.
HIP_FLAGS = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unknown-pragmas",
]


def hipcc():
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    return os.path.join(rocm, "bin", "hipcc")


def source_id(texts):
    """12 hex digits that name the code in the given C++ texts: comments and
    blank space do not count."""
    h = hashlib.sha256()
    for t in texts:
        t = re.sub(r"//[^\n]*|/\*.*?\*/", " ", t, flags=re.S)
        h.update(" ".join(t.split()).encode() + b"\0")
    return h.hexdigest()[:12]


def kernel_id():
    """Names the kernels this tree builds: the library's sources and the flags
    they are compiled with."""
    texts = []
    for f in SOURCES + HEADERS:
        with open(os.path.join(CSRC, f)) as src:
            texts.append(src.read())
    return source_id(texts + [" ".join(HIP_FLAGS)])


def build(verbose=True, asm=False):
    inc = ["-I" + os.path.join(ROOT, "include"), "-I" + CSRC]
    objs = []
    bdir = os.path.join(ROOT, "_build")
    os.makedirs(bdir, exist_ok=True)
    for src in SOURCES:
        obj = os.path.join(bdir, src + ".o")
        lang = ["-x", "hip"]
        cmd = [hipcc()] + HIP_FLAGS + inc + lang + [f'-DOCTOFMM_KERNEL_ID="{kernel_id()}"', "-c",
                                                    os.path.join(CSRC, src), "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.run(cmd, check=True)
        objs.append(obj)
        if asm and src == "octofmm.hip":
            acmd = [hipcc()] + HIP_FLAGS + inc + lang + ["--cuda-device-only", "-S",
                                                         os.path.join(CSRC, src), "-o",
                                                         os.path.join(bdir, src + f".{ARCH}.s")]
            subprocess.run(acmd, check=True)
    tmp = LIB + ".tmp"
    cmd = [hipcc(), "-shared", f"--offload-arch={ARCH}", "-fPIC"] + objs + ["-o", tmp]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    build(asm="--asm" in sys.argv)
