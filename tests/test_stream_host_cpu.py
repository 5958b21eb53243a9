"""What the streaming call makes and keeps, and in which order it moves bytes:
cudec_amd/csrc/stream.cpp over a stand-in for the HIP runtime on the CPU
(tests/stream_host.cpp), where a chunk decodes to its own bytes.

* a context that is kept has its four streams from the start, made one after
  the other; that of a single call has those that the call uses, two at most,
  as much staging, and none of either is left;
* what it keeps for the next call stays within two budgets of staging (1 GiB
  each, or the largest chunk);
* host buffers of one call that lie over each other: what a call of one wave
  gives, every source read before the first byte is written and chunks written
  in order;
* results and bytes of calls of one and of many waves;
* a call whose staging cannot be had leaves no error with the thread."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from tests import libs

BUILD = os.path.join(libs.ROOT, "tests", "_build")
RES = np.dtype([("status", "<i4"), ("reserved", "<u4"), ("bytes_written", "<u8")])
MIB = 1 << 20
HOST = 0


@pytest.fixture(scope="module")
def lib():
    os.makedirs(BUILD, exist_ok=True)
    out = os.path.join(BUILD, "libstream_host.so")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-fPIC",
                    "-shared", "-pthread", "-Wl,-Bsymbolic", "-D__HIP_PLATFORM_AMD__",
                    "-I", os.path.join(libs.ROOT, "include"),
                    "-I", os.path.join(libs.ROOT, "cudec_amd", "csrc"), "-I/opt/rocm/include",
                    "-o", out, os.path.join(libs.ROOT, "tests", "stream_host.cpp")], check=True)
    lib = ctypes.CDLL(out)
    vp, sz = ctypes.c_void_p, ctypes.c_size_t
    lib.cudec_stream_ctx_create.argtypes = [ctypes.POINTER(vp)]
    lib.cudec_stream_ctx_destroy.argtypes = [vp]
    lib.cudec_stream_ctx_destroy.restype = None
    lib.cudec_lz4_decompress_stream_ctx.argtypes = [vp, vp, vp, vp, vp, sz, ctypes.c_int, vp]
    lib.cudec_lz4_decompress_stream.argtypes = [vp, vp, vp, vp, sz, ctypes.c_int, vp]
    lib.host_stream_counts.argtypes = [vp]
    lib.host_stream_counts.restype = None
    lib.host_stream_most_from_here.restype = None
    return lib


def counts(lib):
    c = np.zeros(5, np.uint64)
    lib.host_stream_counts(c.ctypes.data)
    return dict(zip(("streams", "events", "held", "most", "open"), (int(v) for v in c)))


class Context:
    def __init__(self, lib):
        self.lib, self.h = lib, ctypes.c_void_p()
        assert lib.cudec_stream_ctx_create(ctypes.byref(self.h)) == 0

    def run(self, src, sizes, dst, caps):
        """Pointers and sizes as lists; (status, results)."""
        n = len(sizes)
        a = [np.array(v, dtype=np.uint64) for v in (src, sizes, dst, caps)]
        res = np.zeros(n, RES)
        st = self.lib.cudec_lz4_decompress_stream_ctx(
            self.h, *(v.ctypes.data for v in a), n, HOST, res.ctypes.data)
        return st, res

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        self.lib.cudec_stream_ctx_destroy(self.h)


class OneCall:
    """The call that makes a context for itself."""
    def __init__(self, lib):
        self.lib = lib

    def run(self, src, sizes, dst, caps):
        n = len(sizes)
        a = [np.array(v, dtype=np.uint64) for v in (src, sizes, dst, caps)]
        res = np.zeros(n, RES)
        st = self.lib.cudec_lz4_decompress_stream(*(v.ctypes.data for v in a), n, HOST,
                                                  res.ctypes.data)
        return st, res


def plain(ctx, n, size):
    """A call of n chunks of `size` bytes, checked."""
    data = np.random.default_rng(n).integers(0, 256, n * size, dtype=np.uint8)
    out = np.zeros(n * size, np.uint8)
    at = size * np.arange(n, dtype=np.uint64)
    st, res = ctx.run(at + np.uint64(data.ctypes.data), [size] * n,
                      at + np.uint64(out.ctypes.data), [size] * n)
    assert st == 0 and np.all(res["status"] == 0) and np.all(res["bytes_written"] == size)
    assert np.array_equal(out, data)


# chunks of 1 MiB in and out: 24 MiB a wave at least, four waves at once
@pytest.mark.parametrize("n,streams", [(1, 1), (23, 1), (24, 2), (40, 2), (60, 2), (200, 2)])
def test_streams_of_a_context(lib, n, streams):
    before = counts(lib)
    plain(OneCall(lib), n, MIB)
    made = counts(lib)
    assert made["streams"] - before["streams"] == streams
    assert made["events"] - before["events"] == streams
    with Context(lib) as ctx:
        # none made between those of a context
        for _ in range(3):
            made = counts(lib)
            assert made["streams"] - before["streams"] == streams + 4
            assert made["events"] - before["events"] == streams + 4
            plain(ctx, n, MIB)
    assert counts(lib)["open"] == before["open"]


def test_staging_of_a_single_call(lib):
    """Eight waves of 25 MiB in and as much out, two of them in hand."""
    before = counts(lib)
    assert before["held"] == 0
    lib.host_stream_most_from_here()
    plain(OneCall(lib), 200, MIB)
    after = counts(lib)
    assert 100 * MIB <= after["most"] <= 100 * MIB + 65536
    assert after["open"] == before["open"] and after["held"] == 0


@pytest.mark.parametrize("calls", ["AB", "BA", "ABAB", "CAB"])
def test_staging_kept(lib, calls):
    """A: four chunks of 480 MiB of room, a slot each; B: two of 900 MiB, which
    two slots take; C: nine of 100 MiB. (A byte each of input.)"""
    shapes = {"A": (4, 480 * MIB), "B": (2, 900 * MIB), "C": (9, 100 * MIB)}
    src = np.full(16, 7, np.uint8)
    out = np.empty(1920 * MIB, np.uint8)  # hardly touched
    with Context(lib) as ctx:
        for c in calls:
            n, cap = shapes[c]
            st, res = ctx.run([src.ctypes.data] * n, [1] * n,
                              [out.ctypes.data + i * cap for i in range(n)], [cap] * n)
            assert st == 0 and np.all(res["bytes_written"] == 1)
            # tables and results are a few hundred bytes here
            assert counts(lib)["held"] <= 2 * 1024 * MIB + 4096, (calls, c)
        plain(ctx, 60, MIB)


def streams_of(lib, call):
    """Made by a call with a context of its own."""
    before = counts(lib)["streams"]
    call(OneCall(lib))
    return counts(lib)["streams"] - before


# (over its own source or an earlier one, it does not matter when it is written)
@pytest.mark.parametrize("kept", [False, True])
@pytest.mark.parametrize("n,ahead,streams", [(200, 110, 1), (200, 1, 1), (60, 59, 1),
                                             (200, -110, 2), (200, -1, 2), (200, 0, 2)])
def test_outputs_over_sources(lib, n, ahead, streams, kept):
    """Chunk i's output lies where chunk i + ahead's input does."""
    pad = max(0, -ahead)
    arena = np.random.default_rng(5).integers(0, 256, (n + abs(ahead)) * MIB, dtype=np.uint8)
    want = arena.copy()
    for i in range(n):
        want[(i + pad + ahead) * MIB:][:MIB] = arena[(i + pad) * MIB:][:MIB]
    src = [arena.ctypes.data + (i + pad) * MIB for i in range(n)]
    dst = [arena.ctypes.data + (i + pad + ahead) * MIB for i in range(n)]

    def call(ctx):
        st, res = ctx.run(src, [MIB] * n, dst, [MIB] * n)
        assert st == 0 and np.all(res["bytes_written"] == MIB)
    if kept:
        with Context(lib) as ctx:
            call(ctx)
    else:
        assert streams_of(lib, call) == streams
    assert np.array_equal(arena, want)


@pytest.mark.parametrize("step", [0, 1000])
def test_outputs_over_outputs(lib, step):
    """All outputs in one buffer, or each a little further on: the last chunk
    over each byte is what stays."""
    n = 200
    data = np.random.default_rng(6).integers(0, 256, n * MIB, dtype=np.uint8)
    out = np.zeros(MIB + n * step, np.uint8)
    want = out.copy()
    for i in range(n):
        want[i * step:i * step + MIB] = data[i * MIB:(i + 1) * MIB]
    with Context(lib) as ctx:
        st, _ = ctx.run([data.ctypes.data + i * MIB for i in range(n)], [MIB] * n,
                        [out.ctypes.data + i * step for i in range(n)], [MIB] * n)
    assert st == 0 and np.array_equal(out, want)


def test_buffers_side_by_side(lib):
    """Inputs and outputs in turn, in any order, some of them empty: none lies
    over another, and the call overlaps its waves."""
    n = 200
    arena = np.random.default_rng(7).integers(0, 256, 2 * n * MIB, dtype=np.uint8)
    order = np.random.default_rng(8).permutation(n)
    for places in (np.arange(n), order):
        want = arena.copy()
        for p in places:
            want[(2 * p + 1) * MIB:][:MIB] = arena[2 * p * MIB:][:MIB]
        src = [arena.ctypes.data + 2 * int(p) * MIB for p in places] + [0, 0]
        dst = [s + MIB for s in src[:n]] + [0, arena.ctypes.data]

        def call(ctx):
            st, res = ctx.run(src, [MIB] * n + [0, 0], dst, [MIB] * n + [0, 0])
            assert st == 0
        before = arena.copy()
        assert streams_of(lib, call) == 2
        assert np.array_equal(arena, want)
        arena[:] = before
        with Context(lib) as ctx:
            call(ctx)
        assert np.array_equal(arena, want)


@pytest.mark.parametrize("size,cap", [(1, 1 << 44), (1 << 44, 1)])
def test_a_failed_call_leaves_no_error(lib, size, cap):
    """Its status says so; the program's next GPU call did not fail."""
    byte = np.zeros(1, np.uint8)
    before = counts(lib)
    with Context(lib) as ctx:
        for _ in range(2):  # the second finds the context poisoned
            st, res = ctx.run([byte.ctypes.data], [size], [byte.ctypes.data], [cap])
            assert st == libs.DEVICE and np.all(res["status"] == libs.DEVICE)
            assert lib.host_last_error() == 0
    assert counts(lib)["open"] == before["open"] and lib.host_last_error() == 0
    with Context(lib) as ctx:
        plain(ctx, 3, 1000)
