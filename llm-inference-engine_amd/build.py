"""Builds libie_hip.so (the gfx950 paged KV-cache library) in place.

Every source under csrc/ is compiled by hipcc for gfx950 only, as HIP, with
  -ffp-contract=off   fused multiply-adds only where the code writes fmaf, so the
                      RoPE rotation is bit-identical to the reference CPU path;
  -Xclang -target-feature -Xclang -packed-fp32-ops
                      no packed-FP32 VALU instructions (the host pass warns that
                      it does not know the feature; that is harmless).
Objects are compiled in parallel into _build/ and linked into
llm-inference-engine_amd/libie_hip.so, next to this file, and binding/ into the CPython
extension native_calls.so beside it.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
import sysconfig

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
INCLUDE = os.path.join(ROOT, "include")
BUILD = os.path.join(ROOT, "_build", "ie_hip")
LIB = os.path.join(PKG, "libie_hip.so")
ARCH = "gfx950"

CFLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-x", "hip",
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-command-line-argument",
    f"-I{INCLUDE}", f"-I{CSRC}",
]


def hipcc() -> str:
    for cand in (shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (ROCm is required to build libie_hip.so)")


def sources() -> list[str]:
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC)
                  if f.endswith((".hip", ".cpp")))


def _compile(src: str) -> str:
    obj = os.path.join(BUILD, os.path.basename(src) + ".o")
    cmd = [hipcc(), *CFLAGS, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"compile failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    return obj


def build(verbose: bool = False) -> str:
    """Compiles every source (always) and links libie_hip.so; returns its path."""
    os.makedirs(BUILD, exist_ok=True)
    srcs = sources()
    workers = min(len(srcs), max(1, min(8, os.cpu_count() or 1)))
    with cf.ThreadPoolExecutor(workers) as ex:
        objs = list(ex.map(_compile, srcs))
    tmp = LIB + ".tmp"
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs,
           "-L/opt/rocm/lib", "-lrocprofiler-sdk-roctx", "-Wl,-rpath,/opt/rocm/lib"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    build_binding(verbose)
    build_probe(verbose)
    return LIB


BINDING_SRC = os.path.join(PKG, "binding", "native_calls.cpp")
BINDING_LIB = os.path.join(PKG, "native_calls.so")


def build_binding(verbose: bool = False) -> str:
    """The CPython extension that calls libie_hip.so (next to it, found by rpath)."""
    tmp = BINDING_LIB + ".tmp"
    cmd = [shutil.which("g++") or "g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-Wall",
           "-D__HIP_PLATFORM_AMD__", f"-I{INCLUDE}", "-I/opt/rocm/include",
           f"-I{sysconfig.get_paths()['include']}", BINDING_SRC, "-o", tmp, f"-L{PKG}",
           "-l:libie_hip.so", "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"binding build failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, BINDING_LIB)
    if verbose:
        print(f"built {BINDING_LIB}")
    return BINDING_LIB


PROBE_SRC = os.path.join(PKG, "probe", "hbm_probe.hip")
PROBE_LIB = os.path.join(PKG, "libie_probe.so")


def build_probe(verbose: bool = False) -> str:
    """The HBM probes bench.py times next to the decode kernel (measurement only)."""
    tmp = PROBE_LIB + ".tmp"
    cmd = [hipcc(), *CFLAGS, "-shared", PROBE_SRC, "-o", tmp]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"probe build failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, PROBE_LIB)
    if verbose:
        print(f"built {PROBE_LIB}")
    return PROBE_LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
