"""Build the gfx950 hydro library in-tree: ramses2_amd/lib/libramses2_hip.so.

hipcc cross-compiles for gfx950 without a GPU.  Packed-FP32 instructions are
disabled (-packed-fp32-ops) so that float code is emitted as scalar VALU ops.
"""
import os
import shutil
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
LIBNAME = "libramses2_hip.so"
# (source, flags of its own): rh_brick64.hip once per set of brick shapes, the FP64
# brick kernel scheduled for instruction-level parallelism (see there)
MAX_ILP = ["-mllvm", "-amdgpu-sched-strategy=max-ilp"]
UNITS = [("rh_godunov.hip", [])]
UNITS += [("rh_brick64.hip", ["-DRH_SET=%d" % i] + MAX_ILP) for i in range(6)]
UNITS += [(f, []) for f in ("rh_tube.hip", "rh_passes.hip", "rh_abi.hip", "rh_ext.hip", "rh_serve.hip", "rh_amr.hip",
                            "rh_flag.hip")]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("RH_OFFLOAD_ARCH", "gfx950")

FLAGS = ["--offload-arch=" + ARCH, "-O3", "-std=c++17", "-fPIC",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-Wall", "-Wno-unused-function"]


FLANG = os.environ.get("FLANG", "/opt/rocm/lib/llvm/bin/flang")
FSRC = os.path.join(HERE, "fortran")


def lib_path():
    return os.path.join(LIBDIR, LIBNAME)


def fortran_driver_path():
    return os.path.join(LIBDIR, "sod_driver")


def build_fortran():
    """Compile the Fortran binding and the Sod driver against the library
    (flang from ROCm); skipped when flang is not installed."""
    if not os.path.exists(FLANG):
        return None
    mod = os.path.join(LIBDIR, "fmod")
    os.makedirs(mod, exist_ok=True)
    out = fortran_driver_path()
    cmd = [FLANG, "-O2", "-J", mod, "-o", out, os.path.join(FSRC, "hip_interface.f90"),
           os.path.join(FSRC, "sod_driver.f90"), "-L" + LIBDIR, "-lramses2_hip", "-Wl,-rpath,$ORIGIN"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        sys.stderr.write(res.stdout + res.stderr)
        raise RuntimeError("flang failed building the Fortran driver")
    return out


def build(verbose=False, out=None, defines=()):
    """Compile every HIP source into the shared library (always recompiles),
    the objects in parallel."""
    os.makedirs(LIBDIR, exist_ok=True)
    out = out or lib_path()
    tmp = out + ".tmp%d" % os.getpid()
    objdir = tempfile.mkdtemp(prefix="rh_build_")
    jobs = int(os.environ.get("MAX_JOBS", 0)) or len(os.sched_getaffinity(0))

    def compile_unit(i):
        src, own = UNITS[i]
        obj = os.path.join(objdir, "%d.o" % i)
        cmd = [HIPCC] + FLAGS + own + ["-D" + d for d in defines] + ["-c", os.path.join(CSRC, src), "-o", obj]
        return obj, subprocess.run(cmd, cwd=CSRC, capture_output=True, text=True)

    try:
        with ThreadPoolExecutor(max_workers=max(1, min(jobs, len(UNITS)))) as pool:
            done = list(pool.map(compile_unit, range(len(UNITS))))
        res = next((r for _, r in done if r.returncode != 0), None)
        if res is None:
            cmd = [HIPCC, "--offload-arch=" + ARCH, "-shared", "-fPIC", "-o", tmp] + [o for o, _ in done]
            res = subprocess.run(cmd, cwd=CSRC, capture_output=True, text=True)
    finally:
        shutil.rmtree(objdir, ignore_errors=True)
    if res.returncode != 0:
        sys.stderr.write(res.stdout + res.stderr)
        raise RuntimeError("hipcc failed building %s" % LIBNAME)
    if verbose:
        sys.stderr.write("".join(r.stderr for _, r in done))
    os.replace(tmp, out)
    if out == lib_path():
        build_fortran()
    return out


if __name__ == "__main__":
    print(build(verbose=True))
