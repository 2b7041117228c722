"""Runs a piece of Python in a process of its own, with the library bound to tests/fake_hip: host
code only, no GPU.  `fake` is the stand-in's ctypes handle there."""
import atexit
import functools
import os
import shutil
import subprocess
import sys
import tempfile
import textwrap

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes as C, sys
fake = C.CDLL({fake!r}, C.RTLD_GLOBAL)
fake.fake_budget.argtypes = [C.c_size_t]
fake.fake_in_use.restype = C.c_size_t
for f in ("fake_host_mallocs", "fake_dev_mallocs", "fake_dev_copies", "fake_new_left"):
    getattr(fake, f).restype = C.c_long
fake.fake_fail_new.argtypes = fake.fake_pairs.argtypes = [C.c_long]
fake.fake_launched.restype = C.c_char_p
sys.path.insert(0, {root!r})
import numpy as np
from nbodygo_amd import NBodyBatch, NBodyGPU, gen
from nbodygo_amd import _lib as L

def launched():
    return [k for k in fake.fake_launched().decode().split("\\n") if k]
"""


@functools.lru_cache(None)
def fake_path():
    d = tempfile.mkdtemp(prefix="fake_hip_")
    atexit.register(shutil.rmtree, d, True)
    out = os.path.join(d, "libfake_hip.so")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                           "-I", os.path.join(rocm, "include"),
                           os.path.join(ROOT, "tests", "fake_hip", "fake_hip.cpp"), "-o", out])
    return out


def run(body, timeout=120):
    """(exit status, output) of the piece."""
    code = PRELUDE.format(fake=fake_path(), root=ROOT) + textwrap.dedent(body)
    p = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True,
                       timeout=timeout, cwd=ROOT)
    return p.returncode, p.stdout + p.stderr
