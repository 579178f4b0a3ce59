"""Builds libtriton_int_hip.so (gfx950 only) from triton_int_amd/csrc/*.hip with hipcc, and the extension
modules _host.so and _layer_host.so (the host path of launchers and decoder layer, csrc/host*.cpp, against torch's headers)
with g++.

    python -m triton_int_amd.build

Flags that matter for results:
  -ffp-contract=off     every fp32 product / sum in the epilogues is rounded on its own
  -packed-fp32-ops off  no v_pk_*_f32 code generation
"""
from __future__ import annotations

import concurrent.futures
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ_DIR = os.path.join(HERE, "_obj")
LIB_DIR = os.path.join(HERE, "lib")
LIB_PATH = os.path.join(LIB_DIR, "libtriton_int_hip.so")

HOST_MODULES = {"host.cpp": os.path.join(HERE, "_host.so"), "host_layer.cpp": os.path.join(HERE, "_layer_host.so")}

SOURCES = ["lib.hip", "gemm_i8.hip", "rowops.hip", "attention_i8.hip", "quant.hip", "layernorm_fp.hip"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]


def _compile(src: str) -> str:
    obj = os.path.join(OBJ_DIR, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC, *FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "is not a recognized feature" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _build_host(src: str) -> None:
    import torch

    root = os.path.dirname(torch.__file__)
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(HIPCC)))
    if not os.path.isdir(os.path.join(rocm, "include", "hip")):
        rocm = "/opt/rocm"
    # NDEBUG: without it torch's headers bring a thread-local debug counter into each module.  glibc before 2.39 then sends every
    # thread-local access of the libraries loaded earlier (torch, HIP, this library) through __tls_get_addr's slow path until that
    # counter itself is used: 0.3-0.45 us per launch (512 x 768 x 768 linear 6.35 / 6.0 us, three short launches 16.7 / 15.4).
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-DNDEBUG", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *(f"-isystem{d}" for d in (os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
                                      os.path.join(rocm, "include"), sysconfig.get_paths()["include"])),
           os.path.join(CSRC, src), "-o", HOST_MODULES[src], f"-L{os.path.join(root, 'lib')}", "-ltorch_python", "-ltorch_hip", "-ltorch_cpu",
           "-lc10_hip", "-lc10", f"-L{LIB_DIR}", "-l:libtriton_int_hip.so", "-Wl,-rpath,$ORIGIN/lib"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed on {src}:\n{r.stderr}")
    if r.stderr.strip():
        sys.stderr.write(r.stderr + "\n")


def build(verbose: bool = True) -> str:
    os.makedirs(OBJ_DIR, exist_ok=True)
    os.makedirs(LIB_DIR, exist_ok=True)
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, len(SOURCES))) as ex:
        objs = list(ex.map(_compile, SOURCES))
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB_PATH, *objs,
           "-Wl,-rpath,/opt/rocm/lib"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    with concurrent.futures.ThreadPoolExecutor(max_workers=len(HOST_MODULES)) as ex:
        list(ex.map(_build_host, HOST_MODULES))
    if verbose:
        print(f"built {LIB_PATH} ({os.path.getsize(LIB_PATH) // 1024} KiB)")
    return LIB_PATH


if __name__ == "__main__":
    build()
