"""Which plan a launch follows (cudec_amd/csrc/plan.h, built for the CPU): the
default, with its rule for launches of few chunks, until a caller sets one;
then that one, also where it equals the default or lies in the same bin. And
how the launch then runs: directly or through the queue, and from 16 chunks a
wave of its first kernel on through sub-queues."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from tests import libs

BUILD = os.path.join(libs.ROOT, "tests", "_build")
KIB = 1 << 10
DEFAULT = (128 * KIB, 64 * KIB)  # LZ4, Snappy
BLOCKS = 1024


@pytest.fixture(scope="module")
def built():
    os.makedirs(BUILD, exist_ok=True)
    out = os.path.join(BUILD, "libplan_host.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-fPIC", "-shared",
                    "-I", os.path.join(libs.ROOT, "cudec_amd", "csrc"),
                    "-o", out, os.path.join(libs.ROOT, "tests", "plan_host.cpp")], check=True)
    return ctypes.CDLL(out)


@pytest.fixture(scope="module")
def plan(built):
    fn = built.host_plan
    fn.argtypes = [ctypes.c_int, ctypes.c_int] + [ctypes.c_uint64] * 3 + [ctypes.c_void_p] * 2
    fn.restype = None

    def call(fmt, how, threshold, n):
        words, cost = np.zeros(4, np.uint64), ctypes.c_uint64()
        fn(fmt, how, threshold, n, BLOCKS, words.ctypes.data, ctypes.byref(cost))
        return [int(w) >> b & 1 for w in words for b in range(64)], cost.value
    return call


def pipelined_from(bits, cost):
    """Whether the plan pipelines exactly the bins of `cost` and above."""
    octave = cost.bit_length() - 1
    last = 255 - (octave << 2 | (cost >> (octave - 2)) & 3)
    return bits == [1] * (last + 1) + [0] * (255 - last)


@pytest.mark.parametrize("fmt", [0, 1])
def test_default(plan, fmt):
    for n, cost in ((1, 8 * KIB), (2 * BLOCKS, 8 * KIB), (2 * BLOCKS + 1, DEFAULT[fmt])):
        bits, threshold = plan(fmt, 0, 0, n)
        assert pipelined_from(bits, cost) and threshold == DEFAULT[fmt]


@pytest.mark.parametrize("how", [1, 2])
@pytest.mark.parametrize("fmt", [0, 1])
def test_a_chosen_plan_is_followed(plan, fmt, how):
    same_bin = DEFAULT[fmt] * 9 // 8
    for cost in (DEFAULT[fmt], same_bin, 512 * KIB, 8 * KIB):
        for n in (1, 2 * BLOCKS, 2 * BLOCKS + 1, 10 ** 6):
            bits, threshold = plan(fmt, how, cost, n)
            assert pipelined_from(bits, cost)
            assert threshold == (cost if how == 1 else DEFAULT[fmt])


DEFAULT_PLAN, NONE = 1, (1 << 64) - 1
WIDE, ALONE = 768, 2560  # resident blocks beside BLOCKS, on 256 CUs


@pytest.fixture(scope="module")
def launch(built):
    fn = built.host_launch
    fn.argtypes = [ctypes.c_int] + [ctypes.c_uint64] * 5 + [ctypes.c_void_p] * 2
    fn.restype = None

    def call(fmt, threshold, n):
        grids, flags = np.zeros(2, np.uint64), np.zeros(4, np.int32)
        fn(fmt, threshold, n, BLOCKS, 0 if fmt else WIDE, ALONE, grids.ctypes.data,
           flags.ctypes.data)
        return dict(zip(("pipes", "direct", "wide", "many"), map(bool, flags)),
                    grid=int(grids[0]), alone=int(grids[1]))
    return call


@pytest.mark.parametrize("fmt", [0, 1])
def test_sub_queues(launch, fmt):
    """The line lies at 16 chunks a wave of the kernel that comes first, for
    the one that follows it too."""
    for threshold, line in ((DEFAULT_PLAN, 16 * 4 * BLOCKS), (0, 16 * 4 * BLOCKS),
                            (NONE, 16 * 2 * ALONE)):
        for n in (line - 1, line, line + 1, 80_000, 100_003, 10 ** 6):
            r = launch(fmt, threshold, n)
            assert not r["direct"] and r["many"] == (n >= line), (threshold, n)
            assert r["pipes"] == (threshold != NONE)
            assert r["grid"] == (ALONE if threshold == NONE else BLOCKS)
            assert r["alone"] == (ALONE if threshold == DEFAULT_PLAN else 0)


@pytest.mark.parametrize("fmt", [0, 1])
def test_direct_launches(launch, fmt):
    for threshold, most, per in ((DEFAULT_PLAN, BLOCKS, 1), (NONE, 2 * ALONE, 2)):
        for n in (1, 2, 767, 768, 769, most - 1, most, most + 1):
            r = launch(fmt, threshold, n)
            assert r["direct"] == (n <= most)
            if r["direct"]:
                assert r["grid"] == -(-n // per) and r["alone"] == 0
                assert r["wide"] == (fmt == 0 and threshold != NONE and n <= WIDE)
    assert launch(fmt, DEFAULT_PLAN, BLOCKS + 1)["alone"] == (BLOCKS + 2) // 2
