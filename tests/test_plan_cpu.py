"""Which plan a launch follows (cudec_amd/csrc/plan.h, built for the CPU): the
default, with its rule for launches of few chunks, until a caller sets one;
then that one, also where it equals the default or lies in the same bin."""
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
def plan():
    os.makedirs(BUILD, exist_ok=True)
    out = os.path.join(BUILD, "libplan_host.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-fPIC", "-shared",
                    "-I", os.path.join(libs.ROOT, "cudec_amd", "csrc"),
                    "-o", out, os.path.join(libs.ROOT, "tests", "plan_host.cpp")], check=True)
    fn = ctypes.CDLL(out).host_plan
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
