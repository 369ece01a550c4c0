"""Compile the gfx950 causal-product library (hipcc, in-tree).

    python fast-transformers_amd/build.py [--force] [--verbose]

Output: fast_transformers_amd/libftc_causal.so next to the Python package, where
``fast_transformers_amd._native`` loads it, and _ftc_host.so beside it, the Python binding over
the same C ABI (g++ against torch's headers).  hipcc cross-compiles, so no GPU is needed.
"""
import argparse
import glob
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")
OUT = os.path.join(HERE, "fast_transformers_amd", "libftc_causal.so")
HOST_SRC = os.path.join(HERE, "host", "ftc_host.cpp")
HOST_OUT = os.path.join(HERE, "fast_transformers_amd", "_ftc_host.so")
OBJ_DIR = os.path.join(HERE, "build")

# -packed-fp32-ops is switched off on purpose: the compiler must not form
# v_pk_{add,mul,fma}_f32 from scalar float code.
HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument", "-Wno-unknown-warning-option",
    "-I", INCLUDE, "-I", CSRC,
]
# Accumulators in ordinary vector registers: with up to 256 of them in the other file the
# compiler moves the matrix products' sums back and forth in every k-step.
FILE_FLAGS = {"ftc_linear.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"]}


def find_hipcc():
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found")


def sources():
    return sorted(glob.glob(os.path.join(CSRC, "*.hip")))


def headers():
    return sorted(glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(INCLUDE, "*.h")))


def host_command():
    """g++ line of the Python binding: host code only, linked against the library beside it."""
    import sysconfig
    import torch
    root = os.path.dirname(torch.__file__)
    return ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
            "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI,
            "-isystem", os.path.join(root, "include"),
            "-isystem", os.path.join(root, "include", "torch", "csrc", "api", "include"),
            "-isystem", "/opt/rocm/include", "-isystem", sysconfig.get_paths()["include"],
            "-I", INCLUDE, HOST_SRC, "-o", HOST_OUT,
            "-L" + os.path.dirname(OUT), "-l:" + os.path.basename(OUT),
            "-L" + os.path.join(root, "lib"), "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip",
            "-Wl,-rpath,$ORIGIN"]


def stamp(out):
    """Where the recipe that a library was built by is kept."""
    return os.path.join(OBJ_DIR, os.path.basename(out) + ".recipe")


def recipe(cmd):
    """What a library depends on beside its inputs: the command, and for the Python binding the
    versions of torch and Python whose headers it was compiled against."""
    import torch
    versions = [torch.__version__, sys.version] if HOST_OUT in cmd else []
    return "\n".join(list(cmd) + versions)


def stale(out, cmd, inputs):
    """Whether a library is missing, older than an input or built by another recipe."""
    if not (os.path.exists(out) and os.path.exists(stamp(out))):
        return True
    with open(stamp(out)) as f:
        if f.read() != recipe(cmd):
            return True
    return os.path.getmtime(out) < max(os.path.getmtime(i) for i in inputs)


def link(out, cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    with open(stamp(out), "w") as f:
        f.write(recipe(cmd))


def build(force=False, verbose=False, extra_flags=()):
    hipcc = find_hipcc()
    os.makedirs(OBJ_DIR, exist_ok=True)
    newest_header = max(os.path.getmtime(h) for h in headers())
    objs = []
    procs = []
    for src in sources():
        obj = os.path.join(OBJ_DIR, os.path.basename(src) + ".o")
        objs.append(obj)
        fresh = (os.path.exists(obj) and os.path.getmtime(obj) >= os.path.getmtime(src)
                 and os.path.getmtime(obj) >= newest_header)
        if fresh and not force:
            continue
        cmd = [hipcc, "-c", src, "-o", obj] + HIPCC_FLAGS + list(extra_flags) + \
            FILE_FLAGS.get(os.path.basename(src), [])
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((src, subprocess.Popen(cmd)))
    for src, p in procs:
        if p.wait() != 0:
            raise RuntimeError("hipcc failed on %s" % src)
    cmd = [hipcc, "-shared", "-fPIC", "--offload-arch=gfx950", "-fno-gpu-rdc", "-o", OUT] + objs
    if procs or force or stale(OUT, cmd, objs):
        link(OUT, cmd, verbose)
    cmd = host_command()
    if force or stale(HOST_OUT, cmd, [HOST_SRC] + glob.glob(os.path.join(INCLUDE, "*.h"))):
        link(HOST_OUT, cmd, verbose)
    return OUT


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--force", action="store_true")
    ap.add_argument("--verbose", action="store_true")
    a = ap.parse_args()
    print(build(force=a.force, verbose=a.verbose))
