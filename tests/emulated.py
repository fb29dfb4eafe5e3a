"""The engine with its kernels built for the CPU (tests/emulation), for tests
that need no GPU: what a kernel reads and writes out of bounds, and the lists
and results it makes.

While the `emulated` fixture is in use, sgraph calls that library (built once
per session) instead of libsgraph.so; `backend` runs a test on it and, marked
gpu, on the device.
"""
import ctypes
import os
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

import sgraph

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "c-gpustreamgraph_amd")
HERE = os.path.join(ROOT, "tests", "emulation")


def build(out_dir):
    """libsgraph.so's sources against the emulated HIP headers; the path of the library."""
    cxx = shutil.which("clang++", path="/opt/rocm/llvm/bin:" + os.environ.get("PATH", ""))
    if cxx is None:
        pytest.skip("no clang++ to build the kernels for the CPU")
    inc = ["-I", HERE, "-I", os.path.join(ROOT, "include"), "-I", os.path.join(PKG, "csrc"), "-I", os.path.join(PKG, "host")]
    flags = ["-std=c++17", "-O1", "-fPIC", "-w", "-x", "c++"]
    sources = [os.path.join(HERE, "plan.cpp"),  # with sg_engine.hip
               os.path.join(HERE, "emulation.cpp"),
               os.path.join(PKG, "host", "sg_io.cpp"), os.path.join(PKG, "host", "sg_server.cpp")]

    def compile_one(src):
        obj = os.path.join(out_dir, os.path.basename(src) + ".o")
        subprocess.run([cxx, *flags, *inc, "-c", src, "-o", obj], check=True)
        return obj

    with ThreadPoolExecutor() as pool:
        objs = list(pool.map(compile_one, sources))
    so = os.path.join(out_dir, "libsgraph_emulated.so")
    subprocess.run([cxx, "-shared", "-o", so, *objs, "-pthread"], check=True)
    return so


@pytest.fixture(scope="session")
def emulated_path(tmp_path_factory):
    return build(str(tmp_path_factory.mktemp("emulated")))


@pytest.fixture
def emulated(emulated_path, monkeypatch):
    """sgraph on the emulated library (the library, for its emulation_* calls)."""
    monkeypatch.setattr(sgraph, "LIB_PATH", emulated_path)
    monkeypatch.setattr(sgraph, "_lib", None)
    so = ctypes.CDLL(emulated_path)
    so.emulation_replace.restype = ctypes.c_uint64
    so.emulation_reset()
    yield so
    so.emulation_reset()


@pytest.fixture(params=["emulated", pytest.param("device", marks=pytest.mark.gpu)])
def backend(request):
    return request.getfixturevalue("emulated") if request.param == "emulated" else None
