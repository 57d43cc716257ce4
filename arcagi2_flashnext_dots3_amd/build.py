"""Build the gfx950 C-ABI library (libspmla_gfx950.so) in-tree with hipcc.

Every .hip file under csrc/ is compiled to an object (in parallel) and linked into one shared library next to
this file; the Python loader (_lib.py) and the tests load that file. Objects go to _build/ (git-ignored).
csrc/py_call.cpp becomes the extension module _native (the loader's callables; without Python's headers or a C++
compiler it is left out and the loader calls through ctypes).
All HIP code is compiled with packed fp32 instructions disabled (-packed-fp32-ops), see the feature flag below.
"""
import concurrent.futures
import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
REPO = os.path.dirname(HERE)
LIB = os.path.join(HERE, "libspmla_gfx950.so")
NATIVE = os.path.join(HERE, "_native" + sysconfig.get_config_var("EXT_SUFFIX"))
CXX = os.environ.get("CXX", "g++")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
FLAGS = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-Xclang", "-target-feature", "-Xclang",
         "-packed-fp32-ops", "-Wno-unused-command-line-argument", "-I", CSRC, "-I", os.path.join(REPO, "include")]


def _run(cmd):
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l and l.strip())
    if r.returncode != 0:
        raise RuntimeError(f"build failed: {' '.join(cmd)}\n{err}")
    return err


def build_native():
    inc = sysconfig.get_paths()["include"]
    if not os.path.exists(os.path.join(inc, "Python.h")) or shutil.which(CXX.split()[0]) is None:
        if os.path.exists(NATIVE):
            os.remove(NATIVE)
        return None
    tmp = NATIVE + ".tmp"
    _run([*CXX.split(), "-O2", "-std=c++17", "-shared", "-fPIC", "-I", inc, "-I", os.path.join(REPO, "include"),
          os.path.join(CSRC, "py_call.cpp"), "-o", tmp, "-ldl"])
    os.replace(tmp, NATIVE)
    return NATIVE


def build(verbose=False):
    srcs = sorted(f for f in os.listdir(CSRC) if f.endswith(".hip"))
    bdir = os.path.join(REPO, "_build")
    os.makedirs(bdir, exist_ok=True)
    objs = [os.path.join(bdir, f[:-4] + ".o") for f in srcs]
    jobs = min(len(srcs), int(os.environ.get("MAX_JOBS", "8")))
    with concurrent.futures.ThreadPoolExecutor(jobs) as ex:
        futs = [ex.submit(_run, [HIPCC, *FLAGS, "-c", os.path.join(CSRC, s), "-o", o]) for s, o in zip(srcs, objs)]
        for s, f in zip(srcs, futs):
            msg = f.result()
            if verbose and msg:
                print(f"[build] {s}: {msg}", flush=True)
    tmp = LIB + ".tmp"
    _run([HIPCC, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", tmp, *objs])
    os.replace(tmp, LIB)
    build_native()
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
