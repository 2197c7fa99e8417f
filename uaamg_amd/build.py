"""Build the gfx950 HIP library in-tree with hipcc (no JIT cache)."""
import os
import subprocess
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
ROOT = os.path.dirname(HERE)
BUILD_DIR = os.path.join(ROOT, "build")

# -ffp-contract=off: FP64 kernels round exactly like the CPU reference order;
# -packed-fp32-ops off: no v_pk_*_f32 generation.
HIPCC_FLAGS = ["-O3", "-std=c++17", "--offload-arch=gfx950", "-fPIC",
               "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
               "-Wno-unused-result"]


SOURCES = ["engine_f64.hip", "engine_mixed_f64.hip", "engine_f32.hip", "engine_f32_2d.hip", "engine_bf16.hip", "uaamg.hip"]


def build(verbose=False):
    os.makedirs(LIBDIR, exist_ok=True)
    objdir = os.path.join(BUILD_DIR, "obj")
    os.makedirs(objdir, exist_ok=True)
    out = os.path.join(LIBDIR, "libuaamg_hip.so")
    tmp = out + ".tmp"

    def run(cmd):
        if verbose:
            print(" ".join(cmd))
        subprocess.run(cmd, check=True)

    def compile_one(src):
        obj = os.path.join(objdir, src + ".o")
        run(["hipcc"] + HIPCC_FLAGS + ["-c", "-o", obj, os.path.join(CSRC, src)])
        return obj

    # one source per precision, compiled side by side
    with ThreadPoolExecutor(min(len(SOURCES), os.cpu_count() or 1, int(os.environ.get("MAX_JOBS", 16)))) as pool:
        objs = list(pool.map(compile_one, SOURCES))
    run(["hipcc", "--offload-arch=gfx950", "-fPIC", "-shared", "-o", tmp] + objs)
    os.replace(tmp, out)
    return out


def build_host_tools(verbose=False):
    """Compile the C++ host-mirror test program against the built library."""
    os.makedirs(BUILD_DIR, exist_ok=True)
    out = os.path.join(BUILD_DIR, "host_solver_test")
    cmd = ["g++", "-O2", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "include"),
           os.path.join(ROOT, "tests", "cpp", "host_solver_test.cpp"),
           "-L", LIBDIR, "-luaamg_hip", "-Wl,-rpath,$ORIGIN/../uaamg_amd/lib",
           "-Wl,-rpath-link,/opt/rocm/lib", "-o", out]
    if verbose:
        print(" ".join(cmd))
    subprocess.run(cmd, check=True)
    return out
