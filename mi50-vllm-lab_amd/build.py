"""Build libpthdec.so (gfx950) in-tree with hipcc.

    python mi50-vllm-lab_amd/build.py [--save-temps DIR]

The library is the C ABI declared in include/pth_dec.h. Beside it pd_native.so, the Python extension
through which pth_dec.py calls it on torch tensors (host code only, torch's headers). Both are
always rebuilt: hipcc takes about a minute and a stale library is worse than a slow build.
"""
import argparse
import os
import shutil
import subprocess
import sys
import sysconfig
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB_DIR = os.path.join(HERE, "lib")
LIB_PATH = os.path.join(LIB_DIR, "libpthdec.so")
NATIVE_PATH = os.path.join(LIB_DIR, "pd_native.so")
# the C ABI, then the kernels (each file compiles on its own; they share csrc/pd_*.hpp)
SOURCES = [os.path.join(HERE, "csrc", f) for f in
           ("pd_api.hip", "pd_decode.hip", "pd_prefill.hip", "pd_prefill_wide.hip",
            "pd_cache_write.hip")]
KERNEL_SOURCES = SOURCES[1:]
ARCH = "gfx950"

# Packed-FP32 VALU forms are disabled for all device code built here. Symbols are hidden
# unless pd_api.hip exports them (the entry points of include/pth_dec.h).
HIP_FLAGS = [
    "-O3", "-std=c++17", f"--offload-arch={ARCH}", "-fPIC", "-shared", "-fvisibility=hidden",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (ROCm is required to build libpthdec.so)")


def build(save_temps: str | None = None, verbose: bool = False) -> str:
    os.makedirs(LIB_DIR, exist_ok=True)
    tmp = LIB_PATH + ".tmp"
    if save_temps:
        save_temps = os.path.abspath(save_temps)  # the compilers run in it
        os.makedirs(save_temps, exist_ok=True)
    with tempfile.TemporaryDirectory() as objdir:
        # one compiler per source, side by side (the prefill kernels take longest)
        jobs = []
        for src in SOURCES:
            obj = os.path.join(objdir, os.path.basename(src) + ".o")
            cmd = [hipcc(), *(["-save-temps=obj"] if save_temps else []), *(f for f in HIP_FLAGS if f != "-shared"), "-c", "-I",
                   os.path.join(ROOT, "include"), src, "-o", os.path.join(save_temps, os.path.basename(obj)) if save_temps else obj]
            if verbose:
                print(" ".join(cmd), flush=True)
            jobs.append((cmd[-1], subprocess.Popen(cmd, cwd=save_temps, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
        outs = [(obj, p.communicate()[0], p.returncode) for obj, p in jobs]
        for _, text, rc in outs:
            if rc != 0:
                sys.stderr.write(text)
                raise RuntimeError(f"hipcc failed ({rc}) building {LIB_PATH}")
        res = subprocess.run([hipcc(), *HIP_FLAGS, *(obj for obj, _, _ in outs), "-o", os.path.abspath(tmp)],
                             capture_output=True, text=True)
    if res.returncode != 0:
        sys.stderr.write(res.stdout + res.stderr)
        raise RuntimeError(f"hipcc failed ({res.returncode}) building {LIB_PATH}")
    os.replace(tmp, LIB_PATH)
    return LIB_PATH


def build_native() -> str:
    """pd_native.so: pd_python.cpp against the installed torch's headers and libraries."""
    from torch.utils import cpp_extension

    os.makedirs(LIB_DIR, exist_ok=True)
    tmp = NATIVE_PATH + ".tmp"
    rocm = os.path.dirname(os.path.dirname(hipcc()))
    includes = [os.path.join(ROOT, "include"), sysconfig.get_paths()["include"], os.path.join(rocm, "include"),
                *cpp_extension.include_paths()]
    libs = cpp_extension.library_paths()
    cmd = [shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-w",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", *[x for i in includes for x in ("-isystem", i)],
           os.path.join(HERE, "csrc", "pd_python.cpp"), "-o", tmp, *[x for p in libs for x in ("-L" + p,)],
           "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        sys.stderr.write(res.stdout + res.stderr)
        raise RuntimeError(f"g++ failed ({res.returncode}) building {NATIVE_PATH}")
    os.replace(tmp, NATIVE_PATH)
    return NATIVE_PATH


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--save-temps", default=None, help="directory for hipcc -save-temps output")
    ap.add_argument("-v", "--verbose", action="store_true")
    args = ap.parse_args()
    print(build(args.save_temps, args.verbose))
    print(build_native())
