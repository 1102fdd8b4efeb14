"""Builds tests/launch_rules_check.cpp (host compiler only) and loads it."""
import ctypes
import functools
import os
import shutil
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@functools.lru_cache(None)
def rules():
    if shutil.which("g++") is None:
        pytest.skip("no host C++ compiler")
    with tempfile.TemporaryDirectory() as d:
        so = os.path.join(d, "rules.so")
        subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC",
                        "-I", os.path.join(ROOT, "fdk_amd", "csrc"),
                        os.path.join(ROOT, "tests", "launch_rules_check.cpp"), "-o", so], check=True)
        return ctypes.CDLL(so)
