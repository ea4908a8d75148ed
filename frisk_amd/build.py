"""Builds libfrisk_hip.so (HIP kernels + C ABI) for gfx950, in-tree.

    python -m frisk_amd.build          # rebuild everything (HIP library, the device-check library, the frisk_ffi and frisk_launch extensions)
    python -m frisk_amd.build --if-missing   # what is not there yet, the extensions for this interpreter

hipcc cross-compiles without a GPU; the resulting library is loaded from
frisk_amd/lib/ by frisk_amd.runtime.
"""
import argparse
import concurrent.futures
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
OBJDIR = os.path.join(CSRC, "build")
LIB = os.path.join(LIBDIR, "libfrisk_hip.so")
HWCHECK_LIB = os.path.join(LIBDIR, "libfrisk_hwcheck.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
COMMON = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # packed-fp32 instructions are kept out of generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I" + os.path.join(ROOT, "include"), "-I" + CSRC,
    "-Wno-unused-command-line-argument",
]
# (the longest units first)
SOURCES = ["kernels_%s%s.hip" % (t, "" if part == 1 else "_%d" % part) for part in (1, 2, 3, 4) for t in ("f16", "bf16", "i8", "e4m3", "f32") if t != "f32" or part < 3]
SOURCES += ["splitk_reduce.hip", "repack.hip", "tile_ops.hip", "elementwise.hip", "softmax.hip", "attention.hip", "capi.cpp"]


def _compile(src):
    obj = os.path.join(OBJDIR, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC] + COMMON + (["-x", "hip"] if src.endswith(".cpp") else []) + ["-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l and l.strip())
    if r.returncode != 0:
        raise RuntimeError("hipcc failed for %s:\n%s" % (src, err))
    return obj, err


def build(jobs=None, verbose=True):
    os.makedirs(OBJDIR, exist_ok=True)
    os.makedirs(LIBDIR, exist_ok=True)
    jobs = jobs or min(8, os.cpu_count() or 1)
    objs = []
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as pool:
        for obj, err in pool.map(_compile, SOURCES):
            objs.append(obj)
            if verbose and err:
                print(err, file=sys.stderr)
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stderr)
    if verbose:
        print("built", LIB)
    return LIB


def build_hwcheck(verbose=True):
    """libfrisk_hwcheck.so: device-side checks of the MFMA fragment conventions and the MFMA-only loop the benchmark times
    (csrc/hwcheck.hip); used by the GPU tests and bench.py, never by the product library"""
    os.makedirs(LIBDIR, exist_ok=True)
    cmd = [HIPCC] + COMMON + ["-shared", os.path.join(CSRC, "hwcheck.hip"), "-o", HWCHECK_LIB]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("building libfrisk_hwcheck.so failed:\n" + r.stderr)
    if verbose:
        print("built", HWCHECK_LIB)
    return HWCHECK_LIB


FFI_DIR = os.path.join(HERE, "ffi")
EXT_SUFFIX = sysconfig.get_config_var("EXT_SUFFIX")  # (of the interpreter that imports them)
FFI_EXT = os.path.join(HERE, "frisk", "frisk_ffi" + EXT_SUFFIX)
LAUNCH_EXT = os.path.join(HERE, "frisk_launch" + EXT_SUFFIX)
FFI_SOURCES = ["ffi.cpp", "ir.cpp", "runtime.cpp"]


def build_ffi(verbose=True):
    """the `frisk_ffi` CPython extension (IR builder + runtime), host code only"""
    import pybind11
    out = FFI_EXT
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-shared", "-fPIC", "-fvisibility=hidden",
           "-I" + pybind11.get_include(), "-I" + sysconfig.get_paths()["include"], "-I" + os.path.join(ROOT, "include")]
    cmd += [os.path.join(FFI_DIR, f) for f in FFI_SOURCES] + ["-o", out, "-ldl"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("building frisk_ffi failed:\n" + r.stderr)
    if verbose:
        print("built", out)
    return out


def build_launch(verbose=True):
    """the `frisk_launch` CPython extension (the calls of runtime.py that launch kernels), host code only"""
    out = LAUNCH_EXT
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-shared", "-fPIC", "-fvisibility=hidden", "-I" + sysconfig.get_paths()["include"], "-I" + os.path.join(ROOT, "include"),
           os.path.join(FFI_DIR, "launch.cpp"), "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("building frisk_launch failed:\n" + r.stderr)
    if verbose:
        print("built", out)
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--if-missing", action="store_true")
    ap.add_argument("-j", type=int, default=None)
    a = ap.parse_args()
    for path, make in ((LIB, lambda: build(a.j)), (HWCHECK_LIB, build_hwcheck), (FFI_EXT, build_ffi), (LAUNCH_EXT, build_launch)):
        if a.if_missing and os.path.exists(path):
            print("present", path)
        else:
            make()


if __name__ == "__main__":
    main()
