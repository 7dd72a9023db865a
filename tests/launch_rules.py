"""The library's launch rules (csrc/rules.h), built for the host."""
import collections
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


PER_ROW, ROWS, GEMM = 0, 1, 2
FormatPlan = collections.namedtuple("FormatPlan", "kernel waves depth tm tn run_rows")


def format_plan(fmt, out, inp, batch, ws_bytes=64 << 20):
    """The kernel of a block format product; run_rows: batch rows per run of
    the gemm with that scratch."""
    r = (ctypes.c_longlong * 6)()
    lib().rule_format_plan(fmt, out, inp // 32, batch, ctypes.c_longlong(ws_bytes), r)
    return FormatPlan(*r)
