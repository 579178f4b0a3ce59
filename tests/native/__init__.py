"""Programs that run the library's host code on the CPU, HIP's calls replaced (fake_hip.h)."""
import os
import subprocess

from triton_int_amd import build as B

HERE = os.path.dirname(os.path.abspath(__file__))


def build_native(source, directory):
    out = os.path.join(str(directory), os.path.splitext(source)[0])
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(B.HIPCC)))
    rocm = rocm if os.path.isdir(os.path.join(rocm, "include", "hip")) else "/opt/rocm"
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__=1", f"-isystem{rocm}/include", os.path.join(HERE, source), "-o", out,
                    "-rdynamic", f"-L{B.LIB_DIR}", "-l:libtriton_int_hip.so", f"-Wl,-rpath,{B.LIB_DIR}", f"-L{rocm}/lib", f"-Wl,-rpath,{rocm}/lib", "-lamdhip64"],
                   check=True)
    return out
