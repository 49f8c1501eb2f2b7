"""Build recipes (explicit hipcc / g++ command lines, in-tree outputs).

  libmvmc_hip.so   mvmc-rs_amd/_build/   HIP kernels for gfx950 + C ABI + host loader
  liboracle.so     oracle/_build/        CPU FP64 oracle (test infrastructure)

Floating-point contraction is disabled everywhere (-ffp-contract=off): every
parity path relies on unfused multiply/add sequences.  Packed FP32 code
generation is disabled on the device.
"""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
BUILD = os.path.join(HERE, "_build")
ORACLE_BUILD = os.path.join(ROOT, "oracle", "_build")
LIB = os.path.join(BUILD, "libmvmc_hip.so")
ORACLE_LIB = os.path.join(ORACLE_BUILD, "liboracle.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("MVMC_OFFLOAD_ARCH", "gfx950")


def _run(cmd):
    print("+", " ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)


# Translation units of the library: (source, macros).  The Pfaffian kernels
# come in parts (ranges of plane sizes) so that their instances compile side
# by side; the longest object sets the build's time.
UNITS = [("csrc/capi.hip", ()), ("host/model.cpp", ())] + \
    [("csrc/rr_planes.hip", (f"RR_PART={k}",)) for k in range(4)] + \
    [("csrc/rr_planes_c128.hip", (f"RR_PART={k}",)) for k in range(2)]


def object_command(src, macros, obj):
    return [HIPCC, f"--offload-arch={ARCH}", "-O3", "-std=c++20", "-fPIC", "-ffp-contract=off",
            "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
            "-Wno-unused-result"] + [f"-D{d}" for d in macros] + ["-c", "-o", obj, os.path.join(HERE, src)]


def link_command(objs, out):
    return [HIPCC, f"--offload-arch={ARCH}", "-fPIC", "-shared", "-o", out] + objs + \
        ["-L/opt/rocm/lib", "-Wl,-rpath,/opt/rocm/lib"]


def build_library(defines=(), out=None):
    """defines: extra -D macros (MVMC_PHASE_CLOCKS adds the sampling kernel's
    phase clocks); out: output path (default mvmc-rs_amd/_build/libmvmc_hip.so)."""
    out = out or LIB
    os.makedirs(os.path.dirname(out), exist_ok=True)
    jobs = []
    for k, (src, macros) in enumerate(UNITS):
        obj = f"{out}.{k}.o"
        cmd = object_command(src, tuple(macros) + tuple(defines), obj)
        print("+", " ".join(cmd), flush=True)
        jobs.append((obj, cmd, subprocess.Popen(cmd)))
    for _, cmd, p in jobs:
        if p.wait() != 0:
            for _, _, other in jobs:
                other.wait()
            raise subprocess.CalledProcessError(p.returncode, cmd)
    objs = [obj for obj, _, _ in jobs]
    tmp = out + ".tmp"
    _run(link_command(objs, tmp))
    os.replace(tmp, out)
    for obj in objs:
        os.remove(obj)
    return out


def build_oracle():
    os.makedirs(ORACLE_BUILD, exist_ok=True)
    srcs = [os.path.join(ROOT, "oracle", "oracle.cpp"), os.path.join(ROOT, "oracle", "expert.cpp")]
    tmp = ORACLE_LIB + ".tmp"
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-fno-fast-math",
          "-o", tmp] + srcs + ["-lpthread"])
    os.replace(tmp, ORACLE_LIB)
    return ORACLE_LIB


if __name__ == "__main__":
    what = sys.argv[1:] or ["oracle", "lib"]
    if "oracle" in what:
        build_oracle()
    if "lib" in what:
        build_library()
