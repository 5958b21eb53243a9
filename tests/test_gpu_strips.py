"""Groups of many short matches, each of which may wait for the one before it:
they are copied 64 output bytes at a time, sources followed through bytes of
the same strip. LZ4 sequences with literals of 0 to 3 bytes and matches around
a strip's length, at offsets inside, around and beyond a strip and beyond what
a one-wave ring holds; groups that mix them with a longer match; both forms,
few chunks and queued ones; against the oracle. The same for columns of
numbers, few symbols and short periods in all three formats."""
import numpy as np
import pytest
import torch

import cudec_amd
from cudec_amd import workload
from cudec_amd.device import DeviceBatch
from tests.gpu_util import check_against_oracle, gpu
from tests.test_gpu_copy_shapes import last_literals, sequence

pytestmark = gpu

NONE = (1 << 64) - 1
OFFSETS = {"near": (1, 2, 3, 4, 5, 7, 8, 9, 12), "strip": (8, 31, 60, 63, 64, 65, 66, 127, 128, 129),
           "far": (4, 8, 500, 2000, 4000, 4095, 4096, 4097, 8600, 8640, 8700, 11000, 30000)}


def stream(rng, kind):
    out, pos = bytearray(), 0
    for k in range(int(rng.integers(200, 2500))):
        n = int(rng.integers(1, 40)) if k == 0 else int(rng.choice((0, 0, 1, 1, 2, 3)))
        match = int(rng.choice((4, 4, 5, 6, 7, 8, 9, 13, 18)))
        if rng.integers(0, 60) == 0:
            match = int(rng.choice((63, 64, 65, 66, 200, 300)))
        off = min(int(rng.choice(OFFSETS[kind])), pos + n)
        out += sequence(rng.integers(0, 256, n, dtype=np.uint8).tobytes(), off, match)
        pos += n + match
    return bytes(out + last_literals(rng.integers(0, 256, 12, dtype=np.uint8).tobytes())), pos + 12


@pytest.fixture(scope="module", params=list(OFFSETS))
def made(request):
    rng = np.random.default_rng(len(request.param))
    streams, caps = [], []
    for i in range(48):
        s, size = stream(rng, request.param)
        if i % 8 == 5:
            s = s[:int(rng.integers(1, len(s)))]
        streams.append(s)
        caps.append(size - (int(rng.integers(1, 60)) if i % 8 == 3 else 0))
    return request.param, streams, caps


@pytest.mark.parametrize("fill", [0, 1100])
@pytest.mark.parametrize("threshold", [0, NONE])
def test_short_matches(made, threshold, fill):
    kind, streams, caps = made
    st, old = cudec_amd.pipeline_threshold("lz4")
    assert st == 0 and cudec_amd.set_pipeline_threshold("lz4", threshold) == 0
    print(f"[strips] {kind}, threshold {threshold}, {len(streams)} chunks and {fill}", flush=True)
    try:
        res = check_against_oracle("lz4", "tuned", streams + [last_literals(bytes(9))] * fill,
                                   caps + [9] * fill)
    finally:
        assert cudec_amd.set_pipeline_threshold("lz4", old) == 0
    assert np.sum(res["status"][:48] == 0) >= 36


@pytest.mark.parametrize("threshold", [0, NONE])
@pytest.mark.parametrize("fmt", ["lz4", "snappy", "zstd"])
def test_columns(fmt, threshold):
    codec = {"lz4": workload.CODEC_LZ4, "snappy": workload.CODEC_SNAPPY,
             "zstd": workload.CODEC_ZSTD}[fmt]
    if not workload.codec_available(codec):
        pytest.skip("no compressor")
    if fmt == "zstd" and threshold:
        pytest.skip("Zstandard has one form")
    rng = np.random.default_rng(11)
    size, orig = 150_001, []
    for width in (2, 4, 8):
        for step in (1, 3, 50, 70_000):
            a = np.cumsum(rng.integers(0, step + 1, size // width + 1)).astype(f"<i{width}")
            orig.append(a.view(np.uint8)[:size].copy())
    for symbols in (2, 3, 4, 6):
        orig.append(rng.integers(0, symbols, size, dtype=np.uint8))
    for period in (1, 2, 5, 13, 63, 64, 65, 100):
        a = np.tile(rng.integers(0, 256, period, dtype=np.uint8), size // period + 1)[:size]
        a[rng.integers(0, size, 3000)] = 7
        orig.append(a)
    sizes = np.full(len(orig), size, np.uint64)
    data = np.concatenate(orig)
    comp, off, csize = workload.compress(codec, data, workload.offsets_of(sizes), sizes)[:3]
    streams = [comp[int(o):int(o) + int(n)].tobytes() for o, n in zip(off, csize)]
    db = DeviceBatch.from_streams(streams, [size] * len(streams), poison=0x5A)
    db.reset_results()
    print(f"[strips] columns {fmt}, threshold {threshold}", flush=True)
    if fmt == "zstd":
        assert db.run(fmt, "tuned") == 0
    else:
        st, old = cudec_amd.pipeline_threshold(fmt)
        assert st == 0 and cudec_amd.set_pipeline_threshold(fmt, threshold) == 0
        try:
            assert db.run(fmt, "tuned") == 0
        finally:
            assert cudec_amd.set_pipeline_threshold(fmt, old) == 0
    torch.cuda.synchronize()
    res = db.results()
    assert np.all(res["status"] == 0) and np.all(res["bytes_written"] == size)
    for i, got in enumerate(db.outputs(res)):
        assert got == orig[i].tobytes(), i
