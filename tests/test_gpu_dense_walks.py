"""Data whose chains of sequences do not meet when they are walked from wrong
starts: two and four symbols, counters, sorted numbers, short periods. A
pipelined block's parser gives up on segments there and walks from every byte
position, now and then changing over within a window and probing again 15
windows later. LZ4 and Snappy, in the usual windows and (few chunks, LZ4) the
wide ones, with truncations, flipped bytes and short capacities among them,
against the oracle."""
import numpy as np
import pytest

import cudec_amd
from cudec_amd import workload
from tests.gpu_util import check_against_oracle, gpu

pytestmark = gpu

SIZES = (3000, 70_000, 400_000)  # one window, several, more than 16


def mixed(rng, n):
    """Stretches of data that needs it and of data that does not."""
    parts, left = [], n
    while left > 0:
        k = int(rng.integers(500, 60_000))
        parts.append(rng.integers(0, int(rng.choice((2, 4, 16, 256))), k, dtype=np.uint8)
                     if rng.integers(0, 2) else
                     np.tile(rng.integers(0, 256, int(rng.integers(1, 200)), dtype=np.uint8),
                             k)[:k])
        left -= k
    return np.concatenate(parts)[:n]


SHAPES = {
    "two symbols": lambda rng, n: rng.integers(0, 2, n, dtype=np.uint8),
    "four symbols": lambda rng, n: rng.integers(0, 4, n, dtype=np.uint8),
    "int32 counter": lambda rng, n: np.arange(n // 4 + 1, dtype=np.int32).view(np.uint8)[:n].copy(),
    "sorted int64": lambda rng, n: np.cumsum(rng.integers(0, 50, n // 8 + 1)).astype(
        np.int64).view(np.uint8)[:n].copy(),
    "period 100": lambda rng, n: np.tile(rng.integers(0, 256, 100, dtype=np.uint8), n // 100 + 1)[:n],
    "period 5000": lambda rng, n: np.tile(rng.integers(0, 256, 5000, dtype=np.uint8),
                                          n // 5000 + 1)[:n],
    "mixed": mixed,
}


def streams_of(codec, shape):
    rng = np.random.default_rng(len(shape))
    sizes = np.array([s + int(rng.integers(0, 9)) for s in SIZES for _ in range(4)], np.uint64)
    orig = [np.ascontiguousarray(SHAPES[shape](rng, int(s))) for s in sizes]
    comp, off, csize = workload.compress(codec, np.concatenate(orig), workload.offsets_of(sizes),
                                         sizes)[:3]
    streams = [comp[int(o):int(o) + int(n)].tobytes() for o, n in zip(off, csize)]
    caps = [int(s) for s in sizes]
    for i in range(len(streams)):  # of every four: whole, cut, flipped, short of room
        if i % 4 == 1:
            streams[i] = streams[i][:int(rng.integers(1, len(streams[i])))]
        elif i % 4 == 2:
            bad = bytearray(streams[i])
            bad[int(rng.integers(len(bad) // 2, len(bad)))] ^= 1 << int(rng.integers(0, 8))
            streams[i] = bytes(bad)
        elif i % 4 == 3:
            caps[i] -= int(rng.integers(1, 40))
    return streams, caps


@pytest.mark.parametrize("fill", [0, 1100])
@pytest.mark.parametrize("fmt", ["lz4", "snappy"])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_chains_that_do_not_meet(shape, fmt, fill):
    codec = workload.CODEC_LZ4 if fmt == "lz4" else workload.CODEC_SNAPPY
    streams, caps = streams_of(codec, shape)
    last = bytes((0x90,)) + bytes(9) if fmt == "lz4" else bytes((9, 8 << 2)) + bytes(9)
    st, old = cudec_amd.pipeline_threshold(fmt)
    assert st == 0 and cudec_amd.set_pipeline_threshold(fmt, 0) == 0
    print(f"[dense walks] {fmt} {shape}, {len(streams)} chunks and {fill}", flush=True)
    try:
        res = check_against_oracle(fmt, "tuned", streams + [last] * fill, caps + [9] * fill)
    finally:
        assert cudec_amd.set_pipeline_threshold(fmt, old) == 0
    assert np.all(res["status"][0:len(streams):4] == 0) and np.all(res["status"][len(streams):] == 0)
