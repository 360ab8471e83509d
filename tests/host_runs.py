"""Runs a piece of Python against libmf3d_hip.so on a recorded HIP runtime without
a GPU (cpp/hip_stub.cpp), in a process of its own: what the library's host code
allocates, which kernels it chooses and what it does when a call fails.

The code sees ``stub`` (limit, in_use, fail, log, clear), ``lib`` (the C ABI), ``C``
(ctypes), ``_lib``, ``core``, ``ref`` (byref) and ``show(value)``, whose values
``run`` returns."""
from __future__ import annotations

import atexit
import functools
import json
import os
import shutil
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes as C, json, sys
_stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
_stub.stub_log.restype = C.c_char_p
_stub.stub_in_use.restype = C.c_size_t
_stub.stub_limit.argtypes = [C.c_size_t]
from macroflow3d_amd import _lib, core
class stub:
    limit = _stub.stub_limit
    in_use = _stub.stub_in_use
    clear = _stub.stub_clear
    fail = staticmethod(lambda text: _stub.stub_fail(text.encode()))
    log = staticmethod(lambda: [_stub.stub_log(i).decode() for i in range(_stub.stub_log_size())])
lib, ref = _lib.lib(), C.byref
def show(value): print("=" + json.dumps(value), flush=True)
"""


@functools.lru_cache(maxsize=1)
def _stub() -> str:
    """The stub library, built once a process."""
    tmp = tempfile.mkdtemp()
    atexit.register(shutil.rmtree, tmp, ignore_errors=True)
    so = os.path.join(tmp, "hip_stub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC",
                    os.path.join(HERE, "cpp", "hip_stub.cpp"), "-o", so], check=True)
    return so


def run(code: str) -> list:
    """The values that ``code`` showed, in order; raises if it failed."""
    r = subprocess.run([sys.executable, "-c", PRELUDE + code, _stub()], cwd=ROOT,
                       capture_output=True, text=True, timeout=120)
    if r.returncode != 0:
        raise RuntimeError(f"exit {r.returncode}\n{r.stdout}\n{r.stderr}")
    return [json.loads(line[1:]) for line in r.stdout.splitlines() if line.startswith("=")]
