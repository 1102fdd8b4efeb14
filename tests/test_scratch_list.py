"""The list of scratch blocks the library keeps between calls, on the host, over a stand-in
for the HIP runtime (tests/scratch_check.cpp): hand-over between streams and threads, the
bound, no wait in a call, the stream's device, and memory given back."""
import functools
import os
import shutil
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP = os.environ.get("ROCM_PATH", "/opt/rocm") + "/include"


@functools.lru_cache(None)
def program():
    if shutil.which("g++") is None or not os.path.exists(HIP + "/hip/hip_runtime.h"):
        pytest.skip("no host C++ compiler or HIP headers")
    d = tempfile.TemporaryDirectory()
    exe = os.path.join(d.name, "scratch")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-w", "-pthread",
                        "-I", HIP, "-I", os.path.join(ROOT, "include"),
                        "-I", os.path.join(ROOT, "fdk_amd", "csrc"),
                        os.path.join(ROOT, "tests", "scratch_check.cpp"),
                        os.path.join(ROOT, "fdk_amd", "csrc", "capi.cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe, d


@pytest.mark.parametrize("check", ["hand-over", "two streams past the limit", "larger while busy",
                                   "larger beside a smaller", "other device", "out of memory",
                                   "threads"])
def test_scratch_list(check):
    r = subprocess.run([program()[0], check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
