"""How often the chains of a pipelined block's parser fail to meet: the rounds
that its 64 walks take over the windows of 1 MiB LZ4 token chunks, by a model
of the walk, stay below the number after which a window, and the 15 after it,
are walked from every position. Of the token process's first 160 such chunks
these two have the windows that take longest."""
import os
import re

import numpy as np
import pytest

from cudec_amd import workload
from tests import libs

MIB = 1 << 20


def constant(name):
    with open(os.path.join(libs.ROOT, "cudec_amd", "csrc", "tuned.hip")) as f:
        return int(re.search(rf"constexpr uint32_t {name} = (\d+);", f.read()).group(1))


def next_member(s, p):
    """Where the LZ4 sequence at p ends, as if one started there."""
    def at(q):
        return s[q] if q < len(s) else 0

    def extension(q):
        n, e = 0, 255
        while e == 255:
            e = at(q)
            n, q = n + e, q + 1
        return n, q
    token, q = at(p), p + 1
    literals = token >> 4
    if literals == 15:
        more, q = extension(q)
        literals += more
    q += literals + 2
    return extension(q)[1] if token & 15 == 15 else q


def most_rounds(s, segment):
    """Of all windows: the rounds in which some lane walks again."""
    base, most = 0, 0
    while base < len(s):
        limit = len(s) - base
        ends = [min((i + 1) * segment, limit) for i in range(64)]
        entry, exits = [i * segment for i in range(64)], [0] * 64
        moves, rounds = list(range(64)), 0
        while True:
            for i in moves:
                p = entry[i]
                while p < ends[i]:
                    p = next_member(s, base + p) - base
                exits[i] = p
            came = [0] + exits[:-1]
            moved = [i for i in range(64) if came[i] != entry[i]]
            if not moved or came[moved[0]] >= limit:
                break
            rounds += 1
            first, reached = moved[0], came[moved[0]]
            moves = []
            for i in range(64):
                sure = i >= first and reached >= i * segment
                to = reached if sure else came[i]
                if to != entry[i] and (sure or to < ends[i]):
                    entry[i] = to
                    moves.append(i)
        most = max(most, rounds)
        out = exits[-1] if not moved else came[moved[0]]
        if out >= limit:
            break
        base += out
    return most


@pytest.mark.parametrize("seed", [135, 124])
def test_token_windows_meet(seed):
    b = workload.build(workload.CODEC_LZ4, [MIB], [0], [seed])
    rounds = most_rounds(bytes(np.asarray(b.compressed(0)).tobytes()), constant("kSegment"))
    assert rounds == 13
    assert rounds + 4 <= constant("kWalkRounds")
