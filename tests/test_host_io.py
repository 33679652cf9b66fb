"""The host-buffer calls' host code on a stand-in for the HIP runtime
(fake_hip.cpp; no GPU): a call whose results did not come back leaves the
caller's buffers as they were, and a call that is refused leaves nothing on
the stream."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("hip") / "libamdhip64.so.7")
    subprocess.run([f"{ROCM}/llvm/bin/clang++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    f"-I{ROCM}/include", f"-I{ROOT}/fable5_llm_amd/csrc",
                    "-Wl,-soname,libamdhip64.so.7", os.path.join(HERE, "fake_hip.cpp"),
                    "-o", so], check=True)
    return so


@pytest.mark.parametrize("check", ["failed_copies", "refused_calls"])
def test_host_calls(runtime, check):
    r = subprocess.run([sys.executable, os.path.join(HERE, "host_io_check.py"), runtime, check],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
