"""The library's launch rules (csrc/rules.h), built for the host."""
import ctypes
import functools
import os
import subprocess
import tempfile

ROOT = os.path.abspath(os.path.join(os.path.dirname(__file__), ".."))


@functools.lru_cache(maxsize=None)
def lib():
    out = os.path.join(tempfile.mkdtemp(prefix="launch_rules"), "rules.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC",
                           "-I" + os.path.join(ROOT, "welvet.cuda_amd", "csrc"),
                           os.path.join(ROOT, "tests", "host", "rules_check.cpp"), "-o", out])
    return ctypes.CDLL(out)
