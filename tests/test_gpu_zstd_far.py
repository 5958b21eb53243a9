"""Zstandard distances of 2 GiB and more. A single-segment frame's window is
its content size, so an offset code of 31 names distances from 2^31 - 3 to
2^32 - 4 that are decoded (RFC 8878 3.1.1.1.2, 3.1.1.3.2.1.1). The frames are
written by hand: 128 KiB of random bytes, run-length blocks up to just past
the distance, then blocks whose sequences copy from the random bytes, so a
distance that is off by one shows up. What they decode to is computed here, one
sequence after the other.

* explicit distances around 2^31, alone and in batches of more than 64;
* the same taken up again as repeat offsets, by later blocks too, less one,
  and back to near distances;
* distances up to the largest there is, past 4 GiB of output;
* a distance one past the output is refused."""
import random
import struct

import numpy as np
import pytest

from tests import libs
from tests.gpu_util import gpu
from tests.test_zstd_cpu import host, host_decode  # noqa: F401 (host is a fixture)

RAW = 128 << 10
RLE = 128 << 10
FILL = 0x5A
MATCH_CODE, MATCH_BASE, MATCH_BITS = 40, 67, 4  # lengths 67 to 82


def block(kind: int, size: int, body: bytes, last: bool) -> bytes:
    return ((size << 3) | (kind << 1) | last).to_bytes(3, "little") + body


def sequences_block(rng, out, repeats, code, literals, values, last):
    """A compressed block of len(values) sequences of `literals` literals, all
    with offset code `code`; `out` (a Tail) and `repeats` are advanced."""
    lit = bytes(rng.randrange(256) for _ in range(literals * len(values)))
    bits = 1  # the start marker; what is read first lies on top
    for k, value in enumerate(values):
        assert value >> code == 1
        extra = rng.randrange(1 << MATCH_BITS)
        bits = (bits << code) | (value - (1 << code))
        bits = (bits << MATCH_BITS) | extra
        out.put(lit[k * literals:(k + 1) * literals])
        if value > 3:
            d = value - 3
            repeats[:] = [d, repeats[0], repeats[1]]
        else:
            slot = value - 1 + (literals == 0)
            d = repeats[slot] if slot < 3 else repeats[0] - 1
            if slot != 0:
                repeats[:] = [d, repeats[0], repeats[2 if slot == 1 else 1]]
        out.copy(d, MATCH_BASE + extra)
    n = len(lit)
    body = struct.pack("<I", n << 4 | 3 << 2)[:3] + lit
    count = len(values)
    body += bytes([count]) if count < 128 else bytes([(count >> 8) + 128, count & 255])
    body += bytes([0x54, literals, code, MATCH_CODE])  # run-length tables
    body += bits.to_bytes((bits.bit_length() + 7) // 8, "little")
    return block(2, len(body), body, last)


class Tail:
    """The output from `base` on, over the random block and the fill."""

    def __init__(self, raw, base):
        self.raw, self.base, self.tail = raw, base, bytearray()

    def put(self, data):
        self.tail += data

    def copy(self, d, n):
        for _ in range(n):
            p = self.base + len(self.tail) - d
            assert p >= 0
            self.tail.append(self.raw[p] if p < RAW else FILL if p < self.base
                             else self.tail[p - self.base])

    def at(self):
        return self.base + len(self.tail)


def far_frame(seed, base, plan):
    """(frame, raw block, tail): plan(rng, out, last) gives the blocks, as
    (code, literals, [value or function of the output position])."""
    rng = random.Random(seed)
    raw = bytes(rng.randrange(256) for _ in range(RAW))
    blocks = [block(0, RAW, raw, False)]
    left = base - RAW
    while left:
        n = min(left, RLE)
        blocks.append(block(1, n, bytes([FILL]), False))
        left -= n
    out, repeats = Tail(raw, base), [1, 4, 8]
    for i, (code, literals, values) in enumerate(plan):
        made, at = [], out.at()
        for v in values:
            at += literals
            made.append(v(at) if callable(v) else v)
            at += MATCH_BASE  # at least
        blocks.append(sequences_block(rng, out, repeats, code, literals, made,
                                      i + 1 == len(plan)))
    head = struct.pack("<IBQ", 0xFD2FB528, 0xE0, out.at())
    return head + b"".join(blocks), raw, bytes(out.tail)


def to_random(rng):
    """The offset value whose source lies somewhere in the random block (code
    31 if 2^31 + 100 000 bytes or more are there)."""
    place = rng.randrange(200, 90000)
    return lambda at: at - place + 3


def plans():
    rng = random.Random(3)
    g2, g4 = 1 << 31, 1 << 32
    far31 = [g2 + 3 + d for d in (-3, -2, -1, 0, 1, 50, 20000)]
    many = [to_random(rng) for _ in range(70)]
    yield "one", g2 + 60000, [(31, 2, [g2 + 53])]
    yield "around 2^31", g2 + 60000, [(31, 2, far31)]
    yield "a batch and more", g2 + 100000, [(31, 1, many), (31, 0, many[:64])]
    yield "repeats", g2 + 100000, [
        (31, 2, many[:66]),
        (1, 2, [2, 3, 3, 2] * 20),         # the second and the third, in turn
        (1, 0, [2, 3, 3, 2, 3] * 20),      # the third, and the first less one
        (0, 0, [1] * 5),                   # the second
        (0, 3, [1] * 5),                   # the first
        (5, 2, [40, 60, 33] * 25),         # near ones push them out
        (1, 2, [2, 3] * 3),
        (31, 0, [to_random(rng)]),
        (1, 0, [3] * 70),                  # less one, down from a far one
    ]
    yield "past 4 GiB", g4 + 50000, [(31, 2, [g4 - 1, g4 - 2, g4 - 1000, g2 + 5]),
                                     (1, 1, [2, 3] * 40),
                                     (31, 2, [g4 - 1] * 65)]


PLANS = list(plans())


def test_the_frames_by_the_cpu_build(host):  # noqa: F811
    """The expectation itself, held to the frame logic's CPU build."""
    _, base, plan = PLANS[1]
    frame, raw, tail = far_frame(1, base, plan)
    status, out = host_decode(host, frame, base + len(tail))
    assert status == libs.OK
    assert out[:RAW] == raw and out[base:] == tail


@gpu
@pytest.mark.parametrize("case", range(len(PLANS)), ids=[p[0] for p in PLANS])
def test_far_distances(case):
    import torch
    from cudec_amd.device import DeviceBatch
    name, base, plan = PLANS[case]
    print(f"[far distances] {name}: {base} bytes before", flush=True)
    frame, raw, tail = far_frame(case, base, plan)
    total = base + len(tail)
    db = DeviceBatch.from_streams([frame], [total], poison=0xA5)
    db.reset_results()
    assert db.run("zstd") == 0
    torch.cuda.synchronize()
    res = db.results()
    assert int(res["status"][0]) == libs.OK and int(res["bytes_written"][0]) == total
    got = np.frombuffer(db.d_out[base:total].cpu().numpy().tobytes(), np.uint8)
    want = np.frombuffer(tail, np.uint8)
    wrong = np.nonzero(got != want)[0]
    assert wrong.size == 0, (name, int(wrong[0]), int(wrong.size))
    assert db.d_out[:RAW].cpu().numpy().tobytes() == raw
    for lo in range(RAW, base, 1 << 28):
        assert bool((db.d_out[lo:min(base, lo + (1 << 28))] == FILL).all()), lo


@gpu
def test_a_distance_past_the_output_is_refused():
    import torch
    from cudec_amd.device import DeviceBatch
    base = (1 << 31) + 1000
    # two literals, then a distance of the whole output and one byte more; the
    # frame says it copies the random block's first bytes
    frame, _, tail = far_frame(9, base, [(31, 2, [base + 2 + 3])])
    at = frame.rindex(bytes([0x54, 2, 31, MATCH_CODE])) + 4
    bits = int.from_bytes(frame[at:], "little") + (1 << MATCH_BITS)
    bad = frame[:at] + bits.to_bytes(len(frame) - at, "little")
    db = DeviceBatch.from_streams([frame, bad], [base + len(tail)] * 2)
    db.reset_results()
    assert db.run("zstd") == 0
    torch.cuda.synchronize()
    res = db.results()
    assert [int(s) for s in res["status"]] == [libs.OK, libs.CORRUPT]
    assert db.d_out[base:base + len(tail)].cpu().numpy().tobytes() == tail
