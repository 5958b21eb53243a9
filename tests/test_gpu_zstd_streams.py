"""The Zstandard batch entry beside itself and its checksum pass, held to
libzstd alone: two batches at once on two streams, each with scratch of its
own, content checksums with a bit flipped, and batches around one and two
frames for each resident block (2048 on 256 CUs)."""
import random

import numpy as np
import pytest

from cudec_amd import workload
from tests import libs
from tests import zstd_corpus as zc
from tests.gpu_util import gpu

pytestmark = [gpu, pytest.mark.skipif(libs.zstdlib() is None, reason="libzstd absent")]


def test_two_streams_at_once():
    import torch
    from cudec_amd.device import DeviceBatch
    batches = [workload.uneven(n, seed=s, codec=workload.CODEC_ZSTD, octaves=8)
               for n, s in ((2300, 0x51), (300, 0x52), (300, 0x53))]
    dbs = [DeviceBatch(b.comp, b.comp_off, b.comp_size, b.sizes, out_off=b.orig_off)
           for b in batches]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    print("[zstd streams] three batches on two streams", flush=True)
    torch.cuda.synchronize()
    for i, db in enumerate(dbs):
        db.reset_results()
    torch.cuda.synchronize()
    for i, db in enumerate(dbs):  # the third behind the first
        assert db.run("zstd", "tuned", stream=streams[i % 2]) == 0
    torch.cuda.synchronize()
    for b, db in zip(batches, dbs):
        res = db.results()
        assert np.all(res["status"] == libs.OK)
        assert np.array_equal(res["bytes_written"], b.sizes)
        assert np.array_equal(db.output_arena()[:b.orig.size], b.orig)


def test_checksum_bits():
    """A frame with its checksum decodes; with any bit of it flipped it is
    CORRUPT, though its content is right."""
    import torch
    from cudec_amd.device import DeviceBatch
    rng = random.Random(41)
    frames, sizes = [], []
    for size in (1, 3, 31, 32, 33, 200, 4095, 65536, 131073, 300_000):
        data = zc._data(rng.randrange(3), size, rng.getrandbits(63))
        frame = libs.zstd_compress(data, 3, checksum=1)
        frames.append(frame)
        sizes.append(size)
        for bit in range(32):
            bad = bytearray(frame)
            bad[len(bad) - 4 + bit // 8] ^= 1 << (bit % 8)
            frames.append(bytes(bad))
            sizes.append(size)
    db = DeviceBatch.from_streams(frames, sizes)
    db.reset_results()
    print(f"[zstd checksums] {len(frames)} frames", flush=True)
    assert db.run("zstd", "tuned") == 0
    torch.cuda.synchronize()
    status = db.results()["status"].reshape(-1, 33)
    assert np.all(status[:, 0] == libs.OK) and np.all(status[:, 1:] == libs.CORRUPT)


@pytest.mark.parametrize("n", [1, 2, 2047, 2048, 2049, 4096, 4097, 5000])
def test_frames_for_each_block(n):
    import torch
    from cudec_amd.device import DeviceBatch
    rng = np.random.default_rng(n)
    base = workload.build(workload.CODEC_ZSTD, rng.integers(1, 3000, 40), rng.integers(0, 3, 40),
                          rng.integers(1, 1 << 60, 40))
    which = rng.integers(0, 40, n)
    frames = [base.compressed(int(i)) for i in which]
    caps = [int(base.sizes[i]) for i in which]
    want = [base.original(int(i)) for i in which]
    bad = set(range(3, n, 11))
    for i in bad:
        frames[i] = frames[i][:-1]
    db = DeviceBatch.from_streams(frames, caps, poison=0x5A)
    db.reset_results()
    print(f"[zstd blocks] {n} frames", flush=True)
    assert db.run("zstd", "tuned") == 0
    torch.cuda.synchronize()
    res = db.results()
    outs = db.outputs(res)
    for i in range(n):
        assert res["status"][i] == (libs.CORRUPT if i in bad else libs.OK), i
        assert res["bytes_written"][i] == (0 if i in bad else caps[i])
        assert i in bad or outs[i] == want[i], i
