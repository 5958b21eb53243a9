"""The host copy threads (cudec_amd/csrc/host_copy.h) built for the CPU
(tests/host_copy.cpp): every item is done once a round, whatever the number
of threads, and a round allocates nothing, so that it cannot throw while the
streaming call has transfers in flight. Small items go to a thread 64 KiB of
them at a time, large ones one by one."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from tests import libs

BUILD = os.path.join(libs.ROOT, "tests", "_build")


@pytest.fixture(scope="module")
def crew():
    os.makedirs(BUILD, exist_ok=True)
    out = os.path.join(BUILD, "libhost_copy.so")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-fPIC",
                    "-shared", "-pthread", "-Wl,-Bsymbolic",
                    "-I", os.path.join(libs.ROOT, "cudec_amd", "csrc"),
                    "-o", out, os.path.join(libs.ROOT, "tests", "host_copy.cpp")], check=True)
    lib = ctypes.CDLL(out)
    lib.host_copy_rounds.argtypes = [ctypes.c_uint64, ctypes.c_uint64, ctypes.c_uint64,
                                     ctypes.c_void_p]
    lib.host_copy_rounds.restype = ctypes.c_int64
    lib.host_copy_owners.argtypes = [ctypes.c_uint64, ctypes.c_uint64, ctypes.c_void_p]
    lib.host_copy_owners.restype = None
    return lib


@pytest.mark.parametrize("mib", [0, 7, 8, 24, 1024])  # 0, 0, 1, 3 and 7 helpers
@pytest.mark.parametrize("n", [0, 1, 3, 1000])
def test_rounds(crew, mib, n):
    hits = np.zeros(max(n, 1), np.uint32)
    refused = crew.host_copy_rounds(mib << 20, n, 50, hits.ctypes.data)
    assert refused == 0
    assert np.all(hits[:n] == 50)


@pytest.mark.parametrize("n,together", [(500_000, 486), (20_000, 20), (2000, 2)])
def test_small_items_together(crew, n, together):
    """Items of 128 bytes, 3.4 KiB and 33 KiB."""
    owner = np.zeros(n, np.uint64)
    crew.host_copy_owners(64 << 20, n, owner.ctypes.data)
    assert np.all(owner != 0)
    changes = np.flatnonzero(np.diff(owner.astype(np.int64))) + 1
    if len(changes):  # (one thread may have done it all)
        assert np.diff(changes, prepend=0).min() >= together
