"""GPU parity where the pipelined form of the tuned LZ4 and Snappy kernels
changes its way, against the CPU oracle.

* length extensions: a match of two to nine extension bytes is a window
  member, a longer one and a literal of two or more end the window or take
  the exact ladder; each sits at every distance from a window's and the
  chunk's end;
* windows: the first spans 2 KiB of the source and the others 8 KiB, or 64
  equal segments of what is left, and one of more than 1280 members ends
  there: sources around those lengths, made of sequences of 3 to 5 bytes, and
  long literals that jump over whole segments;
* groups: outputs just below and above one group's 2560 bytes, chains of
  short offsets across group borders (members that wait for the group
  before), sources older than the block's LDS history;
* launches: as many chunks as there are resident blocks and more, chunks in
  any order.

Every launch shape decodes every stream, and malformed and short-capacity
copies of it, with the oracle's statuses and bytes.
"""
import numpy as np
import pytest

from tests import libs
from tests.gpu_util import LAUNCHES, check_against_oracle, gpu, oracle_decode
from tests.test_gpu_copy_shapes import last_literals, sequence

pytestmark = gpu


class Writer:
    """An LZ4 stream written sequence by sequence."""

    def __init__(self, seed):
        self.rng = np.random.default_rng(seed)
        self.out, self.pos = bytearray(), 0

    def put(self, lit, off, match):
        lit = lit if self.pos + lit else 1
        off = max(1, min(off, self.pos + lit))
        self.out += sequence(self.rng.integers(0, 256, lit, dtype=np.uint8).tobytes(), off, match)
        self.pos += lit + match

    def done(self, tail=16):
        self.out += last_literals(self.rng.integers(0, 256, tail, dtype=np.uint8).tobytes())
        return bytes(self.out)


def extension_streams():
    for ext in (254, 255, 256, 2 * 255 - 1, 2 * 255, 8 * 255 - 1, 8 * 255, 9 * 255, 9 * 255 + 1,
                20 * 255):
        for before in (0, 1, 120, 680):
            for after in (0, 3, 90):
                w = Writer(ext * 7 + before + after)
                for i in range(before):
                    w.put(int(w.rng.integers(0, 2)), int(w.rng.integers(1, 40)), 4)
                w.put(5, int(w.rng.integers(1, 3000)), 19 + ext)
                w.put(15 + ext, 9, 5)
                for i in range(after):
                    w.put(int(w.rng.integers(0, 4)), int(w.rng.integers(1, 9)), 6)
                yield f"ext{ext}/{before}/{after}", w.done(12 + after % 5)


def window_streams():
    for size in (1, 62, 63, 64, 65, 2047, 2048, 2049, 2700, 8191, 8192, 8193, 10240, 10241, 30000):
        for kind in range(3):
            w = Writer(size * 3 + kind)
            while len(w.out) + 40 < size:
                if kind == 0:
                    w.put(0, int(w.rng.integers(1, 17)), int(w.rng.integers(4, 19)))
                elif kind == 1:
                    w.put(int(w.rng.integers(0, 3)), int(w.rng.integers(1, 60000)),
                          int(w.rng.integers(4, 40)))
                elif w.rng.random() < 0.02:
                    w.put(int(w.rng.integers(100, 1500)), 7, 9)
                else:
                    w.put(int(w.rng.integers(0, 20)), int(w.rng.integers(1, 5000)), 8)
            yield f"window{size}/{kind}", w.done(max(12, min(size - len(w.out) - 1, 14)))


def group_streams():
    for match in (35, 39, 40, 41, 60, 64, 65, 80, 255, 257, 800):
        for off in (1, 3, 15, 16, 17, 40, 1000, 8639, 8641, 16383, 16385, 40000):
            w = Writer(match * 31 + off)
            for i in range(900 * 40 // match):
                near = w.rng.random() < 0.5
                w.put(int(w.rng.integers(0, 3)), int(w.rng.integers(1, 25)) if near else off, match)
            yield f"group{match}/{off}", w.done()


def with_bad_copies(named):
    """The streams at exact capacity, and some truncated, one byte flipped
    or given too little room."""
    rng = np.random.default_rng(99)
    names, streams, caps = [], [], []
    for k, (name, s) in enumerate(named):
        st, out = oracle_decode("lz4", s, 1 << 22)
        assert st == libs.OK, f"the generator wrote an invalid stream: {name}"
        flip = bytearray(s)
        flip[int(rng.integers(0, len(s)))] ^= int(rng.integers(1, 256))
        copies = [(s, len(out)), (s, len(out) + 5), (s[: len(s) - 1 - k % 7], len(out)),
                  (bytes(flip), len(out)), (s, max(0, len(out) - 1 - k % 9))]
        for c, (data, cap) in enumerate(copies if k % 3 == 0 else copies[:1]):
            names.append(f"{name}/{c}")
            streams.append(data)
            caps.append(cap)
    return names, streams, caps


@pytest.mark.parametrize("launch", LAUNCHES)
@pytest.mark.parametrize("make", [extension_streams, window_streams, group_streams])
def test_lz4_edges_exact(make, launch):
    names, streams, caps = with_bad_copies(make())
    print(f"[{make.__name__}] {len(streams)} chunks, {launch}", flush=True)
    check_against_oracle("lz4", launch, streams, caps, names)


@pytest.mark.parametrize("fmt", ["lz4", "snappy"])
@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 2049, 5121])
def test_launch_sizes_exact(fmt, n):
    """The default plan on batches around the number of resident blocks, in
    an order of sizes that no queue sorted."""
    from cudec_amd import workload
    codec = workload.CODEC_LZ4 if fmt == "lz4" else workload.CODEC_SNAPPY
    rng = np.random.default_rng(n)
    base = workload.build(codec, rng.integers(1, 3000, 40), rng.integers(0, 3, 40),
                          rng.integers(1, 1 << 60, 40))
    big = workload.build(codec, rng.integers(60000, 200000, 3), [0, 1, 2], [1, 2, 3])
    streams = [base.compressed(i % 40) for i in range(n)]
    caps = [int(base.sizes[i % 40]) for i in range(n)]
    for k in range(min(3, n)):
        at = int(rng.integers(0, n))
        streams[at], caps[at] = big.compressed(k), int(big.sizes[k])
    if n > 10:
        streams[5] = streams[5][:-1]
        caps[7] -= 1 if caps[7] else 0
    print(f"[launch sizes] {fmt} {n} chunks", flush=True)
    check_against_oracle(fmt, "tuned", streams, caps)


@pytest.mark.parametrize("launch", ["tuned-pipe", "tuned"])
@pytest.mark.parametrize("copies", [1, 768, 769])
def test_lz4_wide_windows_exact(launch, copies):
    """Launches of up to three blocks a CU take windows of 12 KiB of at most
    1920 members: sources around one and two of them behind the first 2 KiB,
    of the shortest sequences and of ones that jump, alone and on both sides
    of the line between the two widths."""
    streams = []
    for size in (12287, 12288, 12289, 14335, 14336, 14337, 26623, 26625, 60000):
        for longest in (4, 19, 300):
            w = Writer(size + longest)
            while len(w.out) + 40 < size:
                near = w.rng.random() < 0.7
                w.put(int(w.rng.integers(0, 2)) if near else int(w.rng.integers(0, 400)),
                      int(w.rng.integers(1, 30 if near else 60000)),
                      int(w.rng.integers(4, longest + 1)))
            streams.append(w.done(max(12, min(size - len(w.out) - 1, 14))))
    caps = [len(oracle_decode("lz4", s, 1 << 22)[1]) for s in streams]
    streams += [streams[1][:-3], streams[7][:9000], streams[11]]
    caps += [caps[1], caps[7], caps[11] - 1]
    if copies > 1:
        streams = [streams[i % len(streams)] for i in range(copies)]
        caps = [caps[i % len(caps)] for i in range(copies)]
    print(f"[wide windows] {len(streams)} chunks, {launch}", flush=True)
    check_against_oracle("lz4", launch, streams, caps)


@pytest.mark.parametrize("fmt", ["lz4", "snappy"])
@pytest.mark.parametrize("big", [0, 1])
@pytest.mark.parametrize("n", [2049, 90000])
def test_queued_batches_with_and_without_a_large_chunk(fmt, n, big):
    """Batches that need the queue, of one and of many chunks a wave, whose
    chunks are all below the pipelining threshold or all but one: the first
    kind goes to the one-wave kernel, the second to the split blocks."""
    from cudec_amd import workload
    codec = workload.CODEC_LZ4 if fmt == "lz4" else workload.CODEC_SNAPPY
    rng = np.random.default_rng(n + big)
    base = workload.build(codec, rng.integers(1, 300, 40), rng.integers(0, 3, 40),
                          rng.integers(1, 1 << 60, 40))
    streams = [base.compressed(i % 40) for i in range(n)]
    caps = [int(base.sizes[i % 40]) for i in range(n)]
    if big:
        large = workload.build(codec, [200000], [0], [1])
        streams[n // 2], caps[n // 2] = large.compressed(0), 200000
    streams[5] = streams[5][:-1]
    caps[7] -= 1
    print(f"[queued] {fmt} {n} chunks, {big} large", flush=True)
    check_against_oracle(fmt, "tuned", streams, caps)


def snappy_element(lit, off, length):
    out = bytearray()
    if lit:
        n = len(lit) - 1
        if n < 60:
            out.append(n << 2)
        else:
            size = (n.bit_length() + 7) // 8
            out.append((59 + size) << 2)
            out += n.to_bytes(size, "little")
        out += lit
    if length:
        out.append(((length - 1) << 2) | 2)
        out += off.to_bytes(2, "little")
    return bytes(out)


@pytest.mark.parametrize("launch", LAUNCHES)
def test_snappy_edges_exact(launch):
    names, streams, caps = [], [], []
    for size in (70, 2048, 2050, 8192, 10245, 30000):
        for kind in range(4):
            rng = np.random.default_rng(size * 5 + kind)
            out, pos = bytearray(), 0
            while len(out) < size:
                n = int(rng.integers(0, 4)) if kind != 2 else int(rng.choice((0, 1, 59, 60, 61, 256, 257, 700)))
                n = n if pos + n else 1
                lit = rng.integers(0, 256, n, dtype=np.uint8).tobytes()
                length = int(rng.integers(1, 65)) if kind != 3 or rng.random() < 0.5 else 0
                off = int(rng.integers(1, (20, 3000, 60000, 9)[kind]))
                out += snappy_element(lit, min(off, pos + n), length)
                pos += n + length
            head, v = bytearray(), pos
            while v >= 128:
                head.append(v & 127 | 128)
                v >>= 7
            head.append(v)
            s = bytes(head + out)
            assert oracle_decode("snappy", s, pos)[0] == libs.OK
            flip = bytearray(s)
            flip[len(s) // 2] ^= 1 + size % 200
            for data, cap in ((s, pos), (s[:-1], pos), (bytes(flip), pos), (s, pos - 1)):
                names.append(f"snappy{size}/{kind}")
                streams.append(data)
                caps.append(cap)
    print(f"[snappy edges] {len(streams)} chunks, {launch}", flush=True)
    check_against_oracle("snappy", launch, streams, caps, names)
