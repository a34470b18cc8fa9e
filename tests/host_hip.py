"""Runs library calls in a child process whose HIP runtime is tests/c/host_hip.cpp (host memory, kernels that
do nothing), so that what the library allocates, gives back and copies can be tested without a GPU."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB = os.path.join(ROOT, "lambda_amd", "liblambda_gpu.so")

PRELUDE = """
import ctypes as C, os, sys, threading
sys.path.insert(0, {root!r})
H = C.CDLL({shim!r}, mode=C.RTLD_GLOBAL)
H.host_hip_live.restype = H.host_hip_pinned.restype = H.host_hip_copies.restype = C.c_uint64
H.host_hip_budget.argtypes = [C.c_uint64]
H.host_hip_copies.argtypes = [C.c_void_p, C.c_uint64]
import numpy as np
from lambda_amd import abi, gpu, scene
def copies():
    "(host address, bytes, kind, thread) of every copy since the last call; kind 1: to the device, 2: to the host"
    a = np.zeros((1 << 16, 4), dtype=np.uint64)
    return a[:H.host_hip_copies(a.ctypes.data, len(a))].astype(np.int64)
live = H.host_hip_live
MB = 1 << 20
dev = gpu.Device(0)
"""


@pytest.fixture(scope="session")
def host_hip(tmp_path_factory):
    """run(code): executes `code` after PRELUDE; it fails by raising."""
    if not os.path.exists(LIB):
        pytest.skip("liblambda_gpu.so is not built")
    shim = str(tmp_path_factory.mktemp("host_hip") / "host_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-o", shim, os.path.join(HERE, "c", "host_hip.cpp")], check=True, capture_output=True)

    def run(code):
        src = PRELUDE.format(root=ROOT, shim=shim) + code + "\nprint('done', flush=True)\nos._exit(0)\n"
        r = subprocess.run([sys.executable, "-c", src], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0 and r.stdout.strip().endswith("done"), r.stdout + r.stderr
    return run
