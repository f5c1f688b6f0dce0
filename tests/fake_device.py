"""Runs a piece of Python against the library on the fake HIP runtime of
tests/fake_hip.cc, in a process of its own."""
import os
import subprocess
import sys
import textwrap
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]
PRELUDE = """
import ctypes as C, sys
fake = C.CDLL({lib!r}, mode=C.RTLD_GLOBAL)  # before the library: its names are found first
fake.fake_log.restype = fake.fake_faults.restype = C.c_char_p
fake.fake_used.restype = C.c_size_t
fake.fake_calls.restype = fake.fake_streams.restype = fake.fake_events.restype = C.c_long
fake.fake_limit.argtypes = [C.c_size_t]
fake.fake_kernel_ms.argtypes = [C.c_char_p, C.c_double]
fake.fake_fail.argtypes = [C.c_char_p, C.c_long, C.c_long, C.c_int]
sys.path[:0] = {path!r}
import numpy as np
import kifmm_amd as K
OUT_OF_MEMORY, DEVICE_LOST = 2, 719
def fail(name, skip=0, count=1, error=DEVICE_LOST):
    fake.fake_fail(name.encode(), skip, count, error)
def log():
    lines = fake.fake_log().decode().splitlines()
    fake.fake_clear_log()
    return lines
def kernels():
    return [ln.split(None, 4) for ln in log() if ln.startswith("kernel ")]
"""


def build(tmp):
    so = Path(tmp) / "libfakehip.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-o", str(so), str(ROOT / "tests" / "fake_hip.cc")], check=True)
    return so


def run(so, code):
    """The code's standard output; fails with its errors, and on a use of what is not live."""
    head = PRELUDE.format(lib=str(so), path=[str(ROOT / "tests"), str(ROOT / "kifmm--hybrid--double-only_amd")])
    tail = "\nassert not fake.fake_faults(), fake.fake_faults().decode()\n"
    r = subprocess.run([sys.executable, "-c", head + textwrap.dedent(code) + tail], capture_output=True, text=True,
                       timeout=120, env=dict(os.environ, OMP_NUM_THREADS="4"))
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout
