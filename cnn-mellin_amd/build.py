#!/usr/bin/env python3
"""Compile libmellin_hip.so for gfx950 with hipcc (cross-compiles without a GPU) and
_mellin_torch.so, the layers' host path for PyTorch, with g++.

    python cnn-mellin_amd/build.py [--force]

Sources: csrc/*.hip and csrc/torch_layer.cpp; output: lib/*.so next to this file.  Packed
FP32 VALU instructions are disabled for all device code.
"""
import glob
import importlib.util
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "lib", "libmellin_hip.so")
TORCH_SRC = os.path.join(CSRC, "torch_layer.cpp")
TORCH_OUT = os.path.join(HERE, "lib", "_mellin_torch.so")
ARCH = "gfx950"

FLAGS = [
    "--offload-arch=" + ARCH, "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-command-line-argument", "-Wno-unknown-warning-option",
]


def sources():
    return sorted(glob.glob(os.path.join(CSRC, "*.hip")))


def up_to_date():
    if not os.path.isfile(OUT) or not os.path.isfile(TORCH_OUT):
        return False
    deps = sources() + [TORCH_SRC] + glob.glob(os.path.join(CSRC, "*.hpp")) + \
        glob.glob(os.path.join(HERE, "..", "include", "*.h")) + [os.path.abspath(__file__)]
    return all(os.path.getmtime(d) <= min(os.path.getmtime(OUT), os.path.getmtime(TORCH_OUT)) for d in deps)


def torch_layer_commands(obj):
    """g++ (compile, link) of the PyTorch host path against the installed torch."""
    torch_dir = os.path.dirname(importlib.util.find_spec("torch").origin)
    inc = [os.path.join(torch_dir, "include"), os.path.join(torch_dir, "include", "torch", "csrc", "api", "include"),
           "/opt/rocm/include", sysconfig.get_paths()["include"]]
    compile_ = ["g++", "-O2", "-std=c++17", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1"] + \
        ["-I" + i for i in inc] + ["-c", TORCH_SRC, "-o", obj]
    link = ["g++", "-shared", obj, "-o", TORCH_OUT, "-L" + os.path.join(torch_dir, "lib"), "-lc10", "-lc10_hip",
            "-ltorch", "-ltorch_cpu", "-ltorch_python", "-L" + os.path.dirname(OUT), "-l:libmellin_hip.so",
            "-Wl,-rpath,$ORIGIN"]
    return compile_, link


def build(force=True, verbose=True):
    if not force and up_to_date():
        return OUT
    os.makedirs(os.path.dirname(OUT), exist_ok=True)
    objdir = os.path.join(HERE, "lib", "obj")
    os.makedirs(objdir, exist_ok=True)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    procs = []
    objs = []
    torch_obj = os.path.join(objdir, "torch_layer.o")
    torch_compile, torch_link = torch_layer_commands(torch_obj)
    if verbose:
        print(" ".join(torch_compile), flush=True)
    procs.append((TORCH_SRC, subprocess.Popen(torch_compile, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)))
    for src in sources():
        obj = os.path.join(objdir, os.path.basename(src)[:-4] + ".o")
        objs.append(obj)
        cmd = [hipcc] + FLAGS + ["-c", src, "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)))
    failed = False
    for src, pr in procs:
        out = pr.communicate()[0].decode()
        out = "\n".join(l for l in out.splitlines() if "packed-fp32-ops" not in l or "error" in l)
        if out.strip() and verbose:
            print(out)
        if pr.returncode != 0:
            print(out)
            failed = True
    if failed:
        raise RuntimeError("compilation failed")
    cmd = [hipcc, "--offload-arch=" + ARCH, "-shared", "-fPIC", "-fno-gpu-rdc"] + objs + ["-o", OUT]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    if verbose:
        print(" ".join(torch_link), flush=True)
    subprocess.check_call(torch_link)
    return OUT


if __name__ == "__main__":
    build(force="--force" in sys.argv or True)
    print("built", OUT)
