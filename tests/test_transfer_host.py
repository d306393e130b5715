"""The copies between host arrays and the device (mpcd_transfer.h) on the CPU,
each direction alone: every byte around the size where a copy is cut into
chunks and at sizes that leave partial ones, and which copies are cut: those
of pageable arrays, while an array the runtime knows (pinned, device or
managed memory) goes to it in one piece, since no copy of the CPU's is faster
than the direct one."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "src_incompressible_openmp_amd", "csrc")
SRC = os.path.join(ROOT, "tests", "transfer_host.cpp")
SO = os.path.join(ROOT, "tests", "_build", "libtransfer_host.so")
DEPS = [SRC, os.path.join(ROOT, "tests", "hip_double", "hip", "hip_runtime.h"), os.path.join(CSRC, "mpcd_transfer.h"),
        os.path.join(CSRC, "mpcd_hip_util.h")]
CHUNK = 2 << 20
CUT_FROM = {1: 10 << 20, 0: 8 << 20, -1: 8 << 20}  # the runtime's own uploads are faster than its downloads
PAGEABLE, PINNED, DEVICE = 0, 1, 2


@pytest.fixture(scope="module")
def one():
    os.makedirs(os.path.dirname(SO), exist_ok=True)
    if not os.path.exists(SO) or any(os.path.getmtime(d) > os.path.getmtime(SO) for d in DEPS):
        subprocess.run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-pthread",
                        "-I" + os.path.join(ROOT, "tests", "hip_double"), "-I" + os.path.join(ROOT, "include"),
                        "-I" + CSRC, SRC, "-o", SO], check=True)
    f = ctypes.CDLL(SO).transfer_one
    f.restype = ctypes.c_longlong
    f.argtypes = [ctypes.c_longlong, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.POINTER(ctypes.c_longlong)]

    def run(n, up, kind, strict=0):
        copies = ctypes.c_longlong()
        return f(n, up, kind, strict, ctypes.byref(copies)), copies.value

    return run


@pytest.mark.parametrize("up", [1, 0, -1], ids=["upload", "download", "download_later"])
@pytest.mark.parametrize("n", [1, 4 * CHUNK - 1, 4 * CHUNK, 4 * CHUNK + 1, 5 * CHUNK - 1, 5 * CHUNK, 5 * CHUNK + 1,
                               8 * CHUNK + 12345, 33 * CHUNK - 8])
def test_pageable(one, n, up):
    for strict in (0, 1):
        bad, copies = one(n, up, PAGEABLE, strict)
        assert bad == 0
        assert copies == (1 if n < CUT_FROM[up] else -(-n // CHUNK))


@pytest.mark.parametrize("up", [1, 0, -1], ids=["upload", "download", "download_later"])
@pytest.mark.parametrize("kind", [PINNED, DEVICE], ids=["pinned", "device"])
def test_registered_goes_direct(one, kind, up):
    for n in (CUT_FROM[up] - 1, CUT_FROM[up], 9 * CHUNK + 77):
        assert one(n, up, kind) == (0, 1)
