"""The Zstandard kernel (a block of two waves a frame) against the CPU build of
the frame logic (tests/zstd_host.cpp) that it shares its parser with: exact
status, size and bytes on every frame, whatever is around.

* the corpus that reaches every block, literals and table mode, with the
  exact capacity, with room and one byte short; hand-made frames; seeded
  mutants;
* sequences written to sit where the kernel changes its way: as many as a
  batch holds (64) and one more or less, literal runs around what a group
  stages, matches around what a group writes, sources in the ring and before
  it;
* literals around the sizes where streams split, of codes that synchronise and
  of codes that hardly do, and damaged ones;
* more frames than there are blocks, from a byte up, at odd output offsets.
"""
import random

import numpy as np
import pytest

from tests import libs
from tests import zstd_corpus as zc
from tests.gpu_util import POISON, gpu
from tests.test_zstd_cpu import host, host_decode  # noqa: F401 (host is a fixture)

pytestmark = [gpu, pytest.mark.skipif(libs.zstdlib() is None, reason="libzstd absent")]


def check(lib, cases):
    """Decodes (name, frame, capacity) in one batch; the statuses."""
    import torch
    from cudec_amd.device import DeviceBatch
    db = DeviceBatch.from_streams([f for _, f, _ in cases], [c for _, _, c in cases],
                                  poison=POISON)
    db.reset_results()
    assert db.run("zstd") == 0
    torch.cuda.synchronize()
    res, arena = db.results(), db.output_arena()
    for i, (name, frame, cap) in enumerate(cases):
        st, out = host_decode(lib, frame, cap)
        assert int(res["status"][i]) == st, name
        if st == libs.OK:
            assert int(res["bytes_written"][i]) == len(out), name
            slot = db.slot(arena, i)
            assert slot[:len(out)].tobytes() == out, name
            assert np.all(slot[len(out):] == POISON), name
    return res["status"]


def test_corpus_capacities(host):  # noqa: F811
    c = zc.corpus()
    cases = [(f"{n}+{d}", f, max(0, len(o) + d)) for n, f, o in c for d in (0, 100, -1)]
    st = check(host, cases)
    assert np.all(st[0::3] == libs.OK) and np.all(st[1::3] == libs.OK)


def test_crafted_and_mutants(host):  # noqa: F811
    cases = [(n, f, c) for n, f, c, _ in zc.crafted()]
    cases += [(n, f, len(d)) for n, f, d in zc.compressor_rejects()]
    frames = [c for c in zc.corpus(max_size=65536) if len(c[1]) > 8]
    cases += zc.mutants(frames, per_frame=12, seed=3)
    assert {libs.OK, libs.CORRUPT, libs.TOO_SMALL} <= set(int(s) for s in check(host, cases))


def written(rng, n, lit, match, back):
    """Bytes to be parsed as n sequences: `lit` new bytes, then `match` bytes
    from `back` before (from what there is, if less), overlapping or not."""
    out = bytearray(rng.integers(0, 256, 64, dtype=np.uint8).tobytes())
    for _ in range(n):
        out += rng.integers(0, 256, lit, dtype=np.uint8).tobytes()
        source = bytes(out[len(out) - min(back, len(out)):])
        out += (source * (match // len(source) + 1))[:match]
    return bytes(out)


SEQUENCES = [(n, lit, match, back)
             for n in (1, 63, 64, 65, 129)
             for lit, match, back in ((1, 5, 40), (0, 200, 7), (12, 30, 5000), (90, 4, 64),
                                      (700, 60, 3000), (720, 2600, 4100), (3, 2555, 12000))]


@pytest.mark.parametrize("level", [1, 9])
def test_sequences_at_the_edges(host, level):  # noqa: F811
    rng = np.random.default_rng(17 + level)
    cases = []
    for n, lit, match, back in SEQUENCES:
        data = written(rng, n, lit, match, back)
        frame = libs.zstd_compress(data, level, checksum=1)
        cases.append((f"{n} of {lit}+{match}@{back}", frame, len(data)))
        cases.append((f"{n} of {lit}+{match}@{back} short", frame, len(data) - 1))
    st = check(host, cases)
    assert np.all(st[0::2] == libs.OK) and np.all(st[1::2] == libs.TOO_SMALL)


def test_wide_sequences_and_repeats(host):  # noqa: F811
    """Sequences of more than 64 bits (far sources, long runs on both sides),
    and copies without literals whose distance steps down by one or returns
    to one of the last three."""
    rng = np.random.default_rng(23)
    far = bytearray(rng.integers(0, 256, 1_700_000, dtype=np.uint8).tobytes())
    for i in range(70):
        far += rng.integers(0, 256, 5000 + 97 * i, dtype=np.uint8).tobytes()
        at = len(far) - 1_600_000 + 1013 * i
        far += far[at:at + 9000 + 131 * i]
    steps = bytearray(rng.integers(0, 256, 4000, dtype=np.uint8).tobytes())
    back = [1500, 700, 300]
    for i in range(600):
        if i % 3 == 0:
            steps += rng.integers(0, 256, i % 5, dtype=np.uint8).tobytes()
        k = int(rng.integers(0, 4))
        d = back[k] if k < 3 else back[0] - 1
        back = [d] + [b for b in back if b != d][:2]
        at = len(steps) - d
        steps += steps[at:at + min(d, 20 + i % 40)]
    cases = []
    for name, data in (("far", bytes(far)), ("steps", bytes(steps))):
        for level in (1, 12, 19):
            cases.append((f"{name} at {level}", libs.zstd_compress(data, level, checksum=1),
                          len(data)))
    assert np.all(check(host, cases) == libs.OK)


def test_literals_at_the_edges(host):  # noqa: F811
    rng = np.random.default_rng(5)
    cases = []
    for size in (60, 61, 255, 256, 257, 700, 1023, 1024, 1025, 2815, 2816, 2817, 16383, 16384,
                 16385, 65535, 131071, 131072, 131073):
        for alphabet in (2, 16, 200):
            w = 1.0 / np.arange(1, alphabet + 1)
            data = rng.choice(alphabet, size, p=w / w.sum()).astype(np.uint8).tobytes()
            cases.append((f"{size} of {alphabet}", libs.zstd_compress(data, 1, checksum=0),
                          size))
        for alphabet in (3, 128, 192):  # codes of one length, or nearly: slow to synchronise
            data = rng.integers(0, alphabet, size, dtype=np.uint8).tobytes()
            cases.append((f"{size} even of {alphabet}", libs.zstd_compress(data, 1, checksum=0),
                          size))
    st = check(host, cases)
    assert np.all(st == libs.OK)
    broken = []
    for name, frame, size in cases:
        for at in (len(frame) - 2, len(frame) - 5, len(frame) // 2):
            bad = bytearray(frame)
            bad[max(at, 0)] ^= 1 << (size % 8)
            broken.append((f"{name} byte {at}", bytes(bad), size))
    assert libs.CORRUPT in set(int(v) for v in check(host, broken))


def test_more_frames_than_blocks(host):  # noqa: F811
    rng = random.Random(29)
    cases = []
    for i in range(4500):
        size = int(2 ** rng.uniform(0, 13))
        data = zc._data(i % 3, size, rng.getrandbits(63))
        cases.append((f"{i}: {size}", libs.zstd_compress(data, (1, 3, 9)[i % 3], checksum=i % 2),
                      size))
    assert np.all(check(host, cases) == libs.OK)
