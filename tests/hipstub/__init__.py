"""Runs the engine's host code on the CPU: a child process loads hipstub.cpp (host-memory stand-ins
of the HIP calls, kernels that do nothing) ahead of libtotem.so and executes a test's program there."""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

PRELUDE = """
import ctypes, sys
import numpy as np
sys.path.insert(0, %r)
sys.modules["torch"] = None          # the engine's own runtime is the stub
stub = ctypes.CDLL(%r, mode=ctypes.RTLD_GLOBAL)
for name in ("in_use", "peak", "in_use_at_info"):
    getattr(stub, "stub_" + name).restype = ctypes.c_size_t
stub.stub_capacity.argtypes = [ctypes.c_size_t]
stub.stub_fill.argtypes = [ctypes.c_size_t, ctypes.c_int]
stub.stub_fail_copy.argtypes = [ctypes.c_long]
for name in ("launches", "pending", "events"):
    getattr(stub, "stub_" + name).restype = ctypes.c_long
stub.stub_widest.restype = ctypes.c_ulonglong
stub.stub_reset_peak.restype = None
from totem_amd import engine, optics
"""


def build(folder):
    so = os.path.join(str(folder), "hipstub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I" + os.path.join(ROCM, "include"), os.path.join(HERE, "hipstub.cpp"), "-o", so], check=True)
    return so


def run(folder, program):
    """Runs the Python program beside the stub; returns what it printed."""
    so = build(folder)
    r = subprocess.run([sys.executable, "-c", PRELUDE % (ROOT, so) + program], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout
