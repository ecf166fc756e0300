"""The library's host code over tests/host_hip.cpp: which kernels a call launches, and with what memory,
checked without a device."""
from __future__ import annotations

import ctypes
import os
import subprocess
from types import SimpleNamespace

from moearc_amd import DeviceView, native

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def build(folder) -> ctypes.CDLL:
    root, out = os.path.dirname(HERE), os.path.join(str(folder), "libmoearc_host.so")
    csrc = os.path.join(root, "moearc_amd", "csrc")
    subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
                    "-I", os.path.join(root, "include"), "-I", csrc, "-I", os.path.join(ROCM, "include"),
                    os.path.join(csrc, "runtime.cpp"), os.path.join(csrc, "kv_cache.cpp"),
                    os.path.join(HERE, "host_hip.cpp"), "-o", out, "-ldl", "-Wl,-Bsymbolic"], check=True)
    lib = ctypes.CDLL(out)
    for name, (res, args) in native.SIGNATURES.items():
        getattr(lib, name).restype, getattr(lib, name).argtypes = res, args
    lib.host_hip_launches.restype = ctypes.c_char_p
    lib.host_hip_largest.argtypes = [ctypes.c_size_t]
    lib.host_hip_allocations.restype = ctypes.c_size_t
    return lib


def launches(lib):
    """[(kernel, grid x, y, z, block)] since the last reset."""
    rows = [r.split() for r in lib.host_hip_launches().decode().splitlines()]
    return [(r[0], *map(int, r[1:])) for r in rows]


def names(lib):
    return [r[0] for r in launches(lib)]


def at(ctx, address: int, nbytes: int) -> DeviceView:
    """A buffer of nbytes at an address of the test's choosing (nothing reads it)."""
    return DeviceView(SimpleNamespace(ctx=ctx, ptr=address, len=nbytes), 0)
