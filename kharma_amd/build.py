"""Build libkharma_amd.so (gfx950) in-tree with hipcc.

    python -m kharma_amd.build [--jobs N]

Objects go to kharma_amd/_build/, the shared library to kharma_amd/libkharma_amd.so.
"""
import argparse
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libkharma_amd.so")
INCLUDE = os.path.abspath(os.path.join(HERE, "..", "include"))

SOURCES = ["kh_flux.hip", "kh_step.hip", "kh_update.hip", "kh_update_f32.hip",
           "kh_update_f64.hip", "kh_adjoint.hip", "kh_mesh.hip", "kh_ct.hip", "kh_capi.cpp", "kh_adjoint_capi.cpp",
           "kh_mesh_capi.cpp", "kh_geom.cpp", "kh_problem.cpp"]
HEADERS = ["kh_device.hpp", "kh_lane_geom.hpp", "kh_step.hpp", "kh_update_geo.hpp", "kh_adjoint.hpp", "kh_internal.hpp", "kh_host.hpp"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("KH_OFFLOAD_ARCH", "gfx950")

# Packed FP32 instructions are disabled for all device code on this platform.
COMMON = ["-std=c++17", "-O3", "-fPIC", f"--offload-arch={ARCH}",
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
          "-Wno-unused-command-line-argument", "-I", CSRC, "-I", INCLUDE]


def _compile(src):
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC] + COMMON + ["-x", "hip", "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"compile {src} failed:\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    return obj


def build(jobs=None, verbose=False):
    os.makedirs(BUILD, exist_ok=True)
    with ThreadPoolExecutor(max_workers=jobs or len(SOURCES)) as ex:
        objs = list(ex.map(_compile, SOURCES))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print("built", LIB)
    return LIB


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=None)
    a = ap.parse_args()
    build(a.jobs, verbose=True)
    sys.exit(0)
