"""Programs that run the library's host code on the stand-in for the HIP
runtime (fake_hip.cpp), each in a process of its own."""
import ctypes
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def build(folder):
    """The stand-in runtime's path, built in folder."""
    so = os.path.join(str(folder), "libamdhip64.so.7")
    subprocess.run([f"{ROCM}/llvm/bin/clang++", "-std=c++17", "-O1", "-shared", "-fPIC",
                    "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include",
                    f"-I{ROOT}/fable5_llm_amd/csrc", "-Wl,-soname,libamdhip64.so.7",
                    os.path.join(HERE, "fake_hip.cpp"), "-o", so], check=True)
    return so


def run(runtime, program, *args, stdin=""):
    """Output of tests/<program> on the runtime."""
    r = subprocess.run([sys.executable, os.path.join(HERE, program), runtime, *args],
                       capture_output=True, text=True, timeout=120, input=stdin)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout.strip()


def load(runtime):
    """(runtime, library), inside such a program: the runtime loaded first
    takes the place of the one that the library names."""
    rt = ctypes.CDLL(runtime, mode=ctypes.RTLD_GLOBAL)
    rt.fake_last_kernel.restype = ctypes.c_char_p
    return rt, ctypes.CDLL(os.path.join(ROOT, "fable5_llm_amd", "libfable5_w4a8.so"))
