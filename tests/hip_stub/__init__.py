"""Programs run in a process of their own, with the CPU stand-in for the HIP
runtime (hip_stub.cpp) in front of libCReaDDyGPU.so."""
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
GXX = shutil.which("g++")
INCLUDE = "/opt/rocm/include"

needs_compiler = pytest.mark.skipif(GXX is None or not os.path.isdir(os.path.join(INCLUDE, "hip")),
                                    reason="g++ or the HIP headers are not available")

PRELUDE = """
import ctypes as C, os, sys
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
import numpy as np
from readdygpu_amd import *
from readdygpu_amd import workloads
stub.stub_name.restype = C.c_char_p
stub.stub_arg.restype = C.c_void_p
stub.stub_arg.argtypes = [C.c_long, C.c_int]
stub.stub_size.restype = C.c_long
stub.stub_size.argtypes = [C.c_void_p]
for f in ("mallocs", "copies", "captures", "graph_launches", "launches"):
    getattr(stub, "stub_" + f).restype = C.c_long
for f in ("name", "fail_malloc", "fail_copy"):
    getattr(stub, "stub_" + f).argtypes = [C.c_long]

def launched(part=""):
    '''(index, name, workgroups, threads, dynamic LDS) of the launches whose name holds `part`'''
    out = []
    d = (C.c_long * 3)()
    for i in range(stub.stub_launches()):
        name = stub.stub_name(i).decode()
        if part in name:
            stub.stub_dims(C.c_long(i), d)
            out.append((i, name, *d))
    return out
"""


def build(tmp):
    so = os.path.join(str(tmp), "libhipstub.so")
    subprocess.run([GXX, "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I" + INCLUDE,
                    os.path.join(HERE, "hip_stub.cpp"), "-o", so], check=True, capture_output=True, timeout=300)
    return so


def run(so, program):
    lib = os.path.join(ROOT, "readdygpu_amd", "libCReaDDyGPU.so")
    if not os.path.exists(lib):
        import __graft_entry__
        __graft_entry__.build()
    r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(program), so, ROOT], capture_output=True,
                       text=True, timeout=300, cwd=ROOT)
    assert r.returncode == 0, (r.stdout + r.stderr)[-4000:]
    return r.stdout
