"""Runs a test's program on the CPU with the library's host code over the
stand-in HIP runtime (fake_hip.cpp): what the host allocates, launches and
copies can be checked without a GPU, also for failures that a GPU run must not
be made to meet."""
from __future__ import annotations

import os
import subprocess
import sys

from conftest import ROOT

# In the program: nv is boxzyhydro_amd.native over the stand-in, fake its
# ctypes handle, launch(f, pinned) has every launch call f(name, grid, block,
# args) and pinned allocations above `pinned` bytes fail.
PRELUDE = """
import ctypes, os, sys, types
import numpy as np
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.modules["torch"] = types.ModuleType("torch")  # its HIP libraries are not for the stand-in
sys.path.insert(0, os.getcwd())
from boxzyhydro_amd import ics, native as nv
from boxzyhydro_amd.params import box_params
import dataclasses
fake.fake_room.restype = fake.fake_bad.restype = ctypes.c_long
fake.fake_room.argtypes = [ctypes.c_void_p]
U3, VPP = ctypes.POINTER(ctypes.c_uint * 3), ctypes.POINTER(ctypes.c_void_p)
FN = ctypes.CFUNCTYPE(None, ctypes.c_char_p, U3, U3, VPP)
keep = []
def launch(f, pinned=2**62):
    keep.append(FN(lambda name, g, b, args: f(name.decode(), list(g.contents), list(b.contents), args)))
    fake.fake_set(keep[-1], ctypes.c_size_t(pinned))
def arg(args, i, kind):
    return ctypes.cast(args[i], ctypes.POINTER(kind)).contents.value
"""


def run(tmp_path, program):
    so = str(tmp_path / "libfake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-w", os.path.join(ROOT, "tests", "fake_hip.cpp"), "-o", so], check=True)
    r = subprocess.run([sys.executable, "-c", PRELUDE + program, so], cwd=ROOT, text=True, capture_output=True)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout
