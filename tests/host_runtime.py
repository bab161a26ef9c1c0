"""Runs a test's code in a process of its own whose engine calls go to
``host_runtime.cc``: no device, no kernel, but the whole host side (checks,
plans, buffers, launches) as a program meets it."""

import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes, os, sys
sys.path.insert(0, {root!r})
host = ctypes.CDLL({lib!r}, mode=ctypes.RTLD_GLOBAL)
host.host_launch.restype = ctypes.c_char_p
host.host_launch.argtypes = [ctypes.c_size_t, ctypes.POINTER(ctypes.c_uint)]
host.host_used.restype = ctypes.c_size_t
host.host_launches.restype = ctypes.c_size_t
host.host_limit.argtypes = [ctypes.c_size_t]
def launches():
    shape = (ctypes.c_uint * 7)()
    return [(host.host_launch(i, shape).decode(), tuple(shape)) for i in range(host.host_launches())]
import numpy as np
import qforte_amd as qf
"""


@pytest.fixture(scope="session")
def on_host(tmp_path_factory):
    """run(code): the code's exit must be clean; its output is returned."""
    lib = str(tmp_path_factory.mktemp("host") / "libhost_runtime.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "host_runtime.cc"), "-o", lib], check=True)

    def run(code, timeout=120):
        text = PRELUDE.format(root=ROOT, lib=lib) + textwrap.dedent(code)
        p = subprocess.run([sys.executable, "-c", text], capture_output=True, text=True, timeout=timeout, cwd=ROOT)
        assert p.returncode == 0, f"exit {p.returncode}\n{p.stdout}\n{p.stderr}"
        return p.stdout

    return run
