"""Build libbolt_hip.so (gfx950) in-tree.

    python bolt.jl_amd/build.py

The library holds the HIP kernels, the C ABI (include/bolt_hip.h) and the
host-side table producers; it is written next to this file.
"""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libbolt_hip.so")
NANFILL_LIB = os.path.join(HERE, "libbolt_hip_nanfill.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

# The solver's, the tables' and the line-of-sight loops span thousands of
# instructions: constants that machine LICM hoists to their tops stay live across
# them and spill registers.
NOLICM = ["-mllvm", "-disable-machine-licm"]
# (object, source, extra flags); the solver is compiled once per scan shape
SOURCES = [("bolt_hip.o", "bolt_hip.hip", NOLICM), ("boltsolve.o", "boltsolve.hip", NOLICM)] + \
          [(f"solve_sr{sr}.o", "solve.hip", NOLICM + [f"-DSOLVE_SR={sr}"]) for sr in (6, 7, 8)] + \
          [("host_tables.o", "host_tables.cpp", []), ("host_api.o", "host_api.cpp", [])]
SOLVERS = ("boltsolve.hip", "solve.hip")


def hip_flags():
    return ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
            # keep hipcc from emitting packed FP32 instructions
            "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
            "-Wno-unused-result", "-I", os.path.join(ROOT, "include")]


def build(verbose=False, nanfill=False):
    """libbolt_hip.so; nanfill=True also builds the debug variant
    libbolt_hip_nanfill.so, whose solver starts every k-mode from a workspace
    filled with NaNs (load it with BOLT_HIP_LIB=<path>)."""
    tmp = os.path.join(HERE, "_build")
    os.makedirs(tmp, exist_ok=True)
    libs, jobs = {LIB: []}, []
    if nanfill:
        libs[NANFILL_LIB] = []
    for name, src, extra in SOURCES:
        cmd = [HIPCC] + hip_flags() + extra
        if src.endswith(".cpp"):
            cmd = [HIPCC, "-x", "c++"] + [f for f in hip_flags() if not f.startswith("--offload-arch")
                                           and f not in ("-Xclang", "-target-feature", "-packed-fp32-ops")] + \
                  (["-ffp-contract=off"] if src == "host_tables.cpp" else [])
        debug = ["-DBOLT_DEBUG_NANFILL"] if src in SOLVERS else None  # the other objects serve both libraries
        for lib, objs in libs.items():
            nan = lib == NANFILL_LIB and debug
            obj = os.path.join(tmp, "nanfill_" + name if nan else name)
            objs.append(obj)
            if lib == NANFILL_LIB and not nan:
                continue
            job = cmd + (debug if nan else []) + ["-c", os.path.join(CSRC, src), "-o", obj]
            if verbose:
                print(" ".join(job), flush=True)
            jobs.append((job, subprocess.Popen(job)))
    for cmd, job in jobs:
        if job.wait():
            raise subprocess.CalledProcessError(job.returncode, cmd)
    for lib, objs in libs.items():
        out_tmp = lib + ".tmp"
        cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", out_tmp] + objs
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.check_call(cmd)
        os.replace(out_tmp, lib)
    return list(libs)[-1]


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv, nanfill="--nanfill" in sys.argv))
