"""Build the gfx950 HIP library libns3d_hip.so in-tree.

    python -m ns3dperiodic_amd.build            # compile (always recompiles)

csrc/ns3d_api.hip exposes the C ABI of include/ns3d.h; the kernels of each grid
length are csrc/ns3d_len.hip, compiled once for each group of lengths.  The
translation units build in parallel, for gfx950 only.
"""
import os
import shutil
import subprocess
import sys
import tempfile
import time
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libns3d_hip.so")

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    "-Wall",
    "-Wno-unused-function",
    # packed FP32 instructions stay off (only ordinary float code is written)
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", os.path.join(ROOT, "include"),
]


def hipcc():
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found: the HIP library cannot be built")
    return exe


# Lengths compiled together: a long plan with a short one, so the groups take similar time.
LENGTH_GROUPS = [(512,), (384, 8), (320, 16), (256, 32), (192, 48), (160, 64), (128, 80), (96,)]


def compile_library(out, flags=(), jobs=8):
    """Compile every translation unit (`jobs` at a time) and link them into `out`."""
    common = [f for f in HIPCC_FLAGS if f != "-shared"] + list(flags)
    with tempfile.TemporaryDirectory() as tmp:
        units = [("ns3d_api.hip", [], "api.o")]
        units += [("ns3d_len.hip", ["-DNS3D_LENGTHS=" + " ".join(f"L({n})" for n in g)], f"len_{g[0]}.o")
                  for g in LENGTH_GROUPS]

        def one(u):
            src, extra, obj = u
            r = subprocess.run([hipcc(), *common, *extra, "-c", os.path.join(CSRC, src), "-o", os.path.join(tmp, obj)],
                               capture_output=True, text=True)
            if r.returncode:
                raise RuntimeError(f"{src} {' '.join(extra)} failed to build:\n{r.stderr[-4000:]}")
            return r.stderr

        with ThreadPoolExecutor(jobs) as ex:
            log = "".join(ex.map(one, units[1:] + units[:1]))
        subprocess.run([hipcc(), "--offload-arch=gfx950", "-fPIC", "-shared", *[os.path.join(tmp, u[2]) for u in units],
                        "-o", out], check=True)
    return log


def build(verbose=True, extra_flags=()):
    tmp = LIB + ".tmp"
    t0 = time.time()
    log = compile_library(tmp, extra_flags, jobs=min(8, os.cpu_count() or 1))
    os.replace(tmp, LIB)
    if verbose:
        if extra_flags:
            print(log)
        print(f"[build] {LIB} ({time.time() - t0:.1f} s)", flush=True)
    build_pattern_ceiling(verbose)
    return LIB


# The access-pattern bandwidth benchmark (a standalone program bench.py runs).
PATTERN_BIN = os.path.join(HERE, "pattern_ceiling")


def build_pattern_ceiling(verbose=True):
    flags = [f for f in HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    tmp = PATTERN_BIN + ".tmp"
    cmd = [hipcc(), *flags, os.path.join(CSRC, "pattern_ceiling.hip"), "-o", tmp]
    if verbose:
        print("[build]", " ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    os.replace(tmp, PATTERN_BIN)
    return PATTERN_BIN


if __name__ == "__main__":
    build(extra_flags=sys.argv[1:])
