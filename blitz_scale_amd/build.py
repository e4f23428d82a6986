"""Compile the gfx950 HIP library in-tree with hipcc.

`python -m blitz_scale_amd.build` writes blitz_scale_amd/lib/libbz_hip.so.  The library is plain
HIP + a C ABI (include/bz_hip.h); it does not link against torch.
"""
import importlib.machinery
import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIB_DIR = os.path.join(HERE, "lib")
LIB_PATH = os.path.join(LIB_DIR, "libbz_hip.so")

SOURCES = [
    "bz_decode_plan.hip",
    "bz_decode.hip",
    "bz_decode_mfma.hip",
    "bz_prefill.hip",
    "bz_page.hip",
    "bz_elementwise.hip",
    "bz_sampler.hip",
    "bz_wire.hip",
    "bz_host.hip",
]

# packed fp32 VALU forms are kept off for every device compile of this library
HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result",
    "-Wno-inline-asm",
]


# bz_decode_mfma.hip: the leading pointers of a kernel's argument list arrive in registers with the wave
# (kernel-argument preload of gfx950), which lets the decode kernel ask for its slot head, and the finishing kernel
# of the decode step for its unit record, while the other arguments are still being fetched: one scalar round trip
# less at the head of each.  A kernel whose first argument is a struct is unaffected.
EXTRA_FLAGS = {
    "bz_decode_mfma.hip": ["-mllvm", "-amdgpu-kernarg-preload-count=4"],
}


def hipcc():
    return os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def build(verbose=True, jobs=8):
    os.makedirs(LIB_DIR, exist_ok=True)
    obj_dir = os.path.join(HERE, "build")
    os.makedirs(obj_dir, exist_ok=True)
    procs = []
    objs = []
    for src in SOURCES:
        path = os.path.join(CSRC, src)
        if not os.path.exists(path):
            continue
        obj = os.path.join(obj_dir, src.replace(".hip", ".o"))
        objs.append(obj)
        cmd = [hipcc(), *HIPCC_FLAGS, *EXTRA_FLAGS.get(src, []), "-I", os.path.join(ROOT, "include"),
               "-I", os.path.join(HERE, "cpp", "kernel"),
               "-c", path, "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
        if len(procs) >= jobs:
            _drain(procs)
    _drain(procs)
    cmd = [hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB_PATH, *objs]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    build_pycall(verbose)
    return LIB_PATH


def build_pycall(verbose=True):
    """The extension module through which kernel.py calls the library (host code only), for the interpreter that runs this.
    Optional: without a C++ compiler or this Python's headers (3.9 or newer) the calls go through ctypes, at 1 to 3 us more each."""
    path = os.path.join(LIB_DIR, "bz_pycall" + importlib.machinery.EXTENSION_SUFFIXES[0])
    cxx, include = os.environ.get("CXX", "g++"), sysconfig.get_paths()["include"]
    if sys.version_info < (3, 9) or not shutil.which(cxx.split()[0]) or not os.path.exists(os.path.join(include, "Python.h")):
        if os.path.exists(path):
            os.remove(path)  # (of an earlier build: its list of calls may be another one)
        print(f"bz_pycall: no C++ compiler ({cxx}) or no Python headers ({include}); calls go through ctypes", flush=True)
        return None
    cmd = [*cxx.split(), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Wno-missing-field-initializers",
           "-I", include, "-I", os.path.join(ROOT, "include"), os.path.join(CSRC, "bz_pycall.cpp"), "-o", path]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    return path


PROBE_SRC = os.path.join(HERE, "probes", "mfma_ceiling.hip")
PROBE_BIN = os.path.join(HERE, "probes", "mfma_ceiling")


def build_probes(verbose=True):
    """The stand-alone measurement program behind `bench.py --workload MFMA_CEILING` (no part of the library)."""
    cmd = [hipcc(), *[f for f in HIPCC_FLAGS if f != "-fPIC"], PROBE_SRC, "-o", PROBE_BIN]
    if verbose:
        print(" ".join(cmd), flush=True)
    out = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    text = "\n".join(l for l in out.stdout.splitlines() if "packed-fp32-ops" not in l)
    if out.returncode != 0:
        raise RuntimeError("hipcc failed on the probe:\n" + text)
    return PROBE_BIN


def _drain(procs):
    failed = []
    for src, p in procs:
        out, _ = p.communicate()
        # the host pass does not know the packed-fp32 target feature and says so: harmless
        out = "\n".join(l for l in out.splitlines() if "packed-fp32-ops" not in l)
        if p.returncode != 0:
            failed.append((src, out))
        elif out.strip():
            print(out)
    procs.clear()
    if failed:
        for src, out in failed:
            sys.stderr.write(f"--- {src} failed ---\n{out}\n")
        raise RuntimeError("hipcc failed for: " + ", ".join(s for s, _ in failed))


if __name__ == "__main__":
    print(build())
