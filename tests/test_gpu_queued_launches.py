"""Launches that need the work queue, whatever makes them: more chunks than
resident blocks and waves (1024 and 5120 on 256 CUs), decoded through every
entry that builds or follows the queue, against the plain form chunk by
chunk: statuses, sizes, bytes and the poison beyond them.

* plans that pipeline every chunk, some, none of those there are (the one-wave
  kernel follows an empty launch) and none at all;
* the batch entry, the parse-only build (no byte written), the allocation-free
  entry, whose second call is smaller and must not see the first's queue, and
  both decoding entries captured into a graph, where the scratch is a graph
  allocation or the fixed array;
* the one-wave kernel around one and two chunks for each of its waves, and
  batches with chunks in every cost bin there is from nothing to 4 MiB;
* the streams of the copy, slow-sequence and chain tests, which have a block
  each there and so the wide windows, in the usual ones;
* matches on both sides of the piece that a pipelined block expands at once
  (15 328 bytes) and of what a group holds (2058), at offsets around what its
  ring and its history hold, in the usual windows and in the wide ones."""
import numpy as np
import pytest
import torch

import cudec_amd
from cudec_amd import workload
from cudec_amd.device import DeviceBatch
from cudec_amd.graph import CapturedLaunch
from tests import libs
from tests.gpu_util import check_against_oracle, gpu, oracle_decode
from tests.test_gpu_copy_shapes import last_literals, sequence, shaped  # noqa: F401
from tests.test_gpu_slow_sequences import slow_chunks  # noqa: F401
from tests.test_gpu_walk_edges import chains  # noqa: F401

pytestmark = gpu

POISON = 0x5A
SIZES = (6000, 5300)
NONE = (1 << 64) - 1
THRESHOLDS = (0, 16 << 10, 1 << 40, NONE)


class plan_by_threshold:
    def __init__(self, fmt, threshold):
        self.fmt, self.threshold = fmt, threshold

    def __enter__(self):
        st, self.old = cudec_amd.pipeline_threshold(self.fmt)
        assert st == 0
        assert cudec_amd.set_pipeline_threshold(self.fmt, self.threshold) == 0

    def __exit__(self, *exc):
        assert cudec_amd.set_pipeline_threshold(self.fmt, self.old) == 0


def snapshot(db):
    torch.cuda.synchronize()
    return db.results().copy(), db.d_out.clone()


def clear(db):
    db.d_out.fill_(POISON)
    db.reset_results()


def arguments(db):
    return (db.src_ptrs.data_ptr(), db.src_sizes.data_ptr(), db.dst_ptrs.data_ptr(),
            db.dst_caps.data_ptr(), db.n, db.d_results.data_ptr())


def noalloc(db, stream=None):
    return cudec_amd.lib().cudec_mi355x_lz4_decompress_batch_noalloc(
        *arguments(db), stream.cuda_stream if stream else None)


@pytest.fixture(scope="module")
def batches():
    """Per format, batches of SIZES chunks with what the plain form gives."""
    out = {}
    for fmt, codec in (("lz4", workload.CODEC_LZ4), ("snappy", workload.CODEC_SNAPPY)):
        b = workload.uneven(SIZES[0], seed=0x9E0E, codec=codec, min_size=1024, octaves=5)
        made = []
        for n in SIZES:
            comp = [b.compressed(i) for i in range(n)]
            caps = [int(s) for s in b.sizes[:n]]
            for i in range(n % 7, n, 9):
                comp[i] = comp[i][:-1]
            for i in range(n % 5, n, 13):
                caps[i] = max(caps[i] - 1, 0)
            db = DeviceBatch.from_streams(comp, caps, poison=POISON)
            db.reset_results()
            assert db.run(fmt, "plain") == 0
            made.append((db, snapshot(db)))
        out[fmt] = made
    return out


# Where a chunk fails, its destination's bytes are not specified; the others'
# are, and so is the room behind them.
def check(db, want, what):
    got = snapshot(db)
    assert np.array_equal(got[0], want[0]), what
    ok = torch.from_numpy((want[0]["status"] == 0)).cuda()
    sizes = torch.from_numpy(db.caps.astype(np.int64)).cuda()
    keep = torch.repeat_interleave(ok, sizes)
    total = keep.numel()
    assert bool(((got[1][:total] == want[1][:total]) | ~keep).all()), what
    assert bool((want[0]["status"] == 0).any()) and bool((want[0]["status"] != 0).any())


@pytest.mark.parametrize("fmt", ["lz4", "snappy"])
@pytest.mark.parametrize("threshold", THRESHOLDS)
def test_batch_and_parse(batches, fmt, threshold):
    with plan_by_threshold(fmt, threshold):
        for db, want in batches[fmt]:
            print(f"[queued] {fmt} {db.n} chunks, threshold {threshold}", flush=True)
            clear(db)
            assert db.run(fmt, "tuned") == 0
            check(db, want, "batch")
            clear(db)
            assert cudec_amd.lib().cudec_mi355x_parse_batch(cudec_amd.FORMAT_CODE[fmt],
                                                            *arguments(db), None) == 0
            res, out = snapshot(db)
            assert np.array_equal(res, want[0]) and bool((out == POISON).all())


@pytest.mark.parametrize("threshold", THRESHOLDS)
def test_allocation_free(batches, threshold):
    with plan_by_threshold("lz4", threshold):
        for db, want in batches["lz4"]:
            print(f"[queued] allocation-free {db.n} chunks, threshold {threshold}", flush=True)
            clear(db)
            assert noalloc(db) == 0
            check(db, want, "allocation-free")


@pytest.mark.parametrize("entry", ["lz4", "snappy", "noalloc"])
@pytest.mark.parametrize("threshold", THRESHOLDS)
def test_graph_replays(batches, entry, threshold):
    fmt = "lz4" if entry == "noalloc" else entry
    (db, want), (other, other_want) = batches[fmt]
    s = torch.cuda.Stream()

    def launch():
        return noalloc(db, s) if entry == "noalloc" else db.run(fmt, "tuned", stream=s)

    print(f"[queued] graph of {entry}, {db.n} chunks, threshold {threshold}", flush=True)
    torch.cuda.synchronize()
    with plan_by_threshold(fmt, threshold):
        with CapturedLaunch(launch, s) as g:
            for k in range(3):
                with torch.cuda.stream(s):
                    clear(db)
                g.replay()
                s.synchronize()
                check(db, want, f"replay {k}")
                # the program's own eager work in between
                clear(other)
                assert other.run(fmt, "tuned") == 0
                check(other, other_want, f"eager launch after replay {k}")


PIECE = 16384 - 1024 - 32
MATCHES = (273, 274, 275, 2057, 2058, 2059, PIECE - 1, PIECE, PIECE + 1, 2 * PIECE - 1, 2 * PIECE,
           2 * PIECE + 1, 50000)
OFFSETS = (1, 2, 3, 7, 15, 16, 17, 64, 999, 1023, 1024, 1025, 8639, 8640, 8641, 16383, 16384,
           16385, 40000, 65535)


def pieces_stream(seed):
    rng = np.random.default_rng(seed)
    out, pos = bytearray(), 0
    for k in range(int(rng.integers(3, 9))):
        n = int(rng.choice((1, 4, 17, 63, 64, 65, 300, 5000))) if k == 0 or rng.integers(0, 2) else 0
        off = max(1, min(int(rng.choice(OFFSETS)), pos + n))
        match = int(rng.choice(MATCHES))
        out += sequence(rng.integers(0, 256, n, dtype=np.uint8).tobytes(), off, match)
        pos += n + match
        for _ in range(int(rng.choice((0, 1, 70)))):
            # short ones right after, from near and from before the match
            off = int(rng.integers(1, min(pos + 3, 20000) + 1))
            out += sequence(rng.integers(0, 256, 3, dtype=np.uint8).tobytes(), off, 37)
            pos += 40
    return bytes(out + last_literals(rng.integers(0, 256, 13, dtype=np.uint8).tobytes()))


@pytest.mark.parametrize("fill", [0, 1100])  # a block each; queued
@pytest.mark.parametrize("threshold", [0, NONE])
def test_pieces_of_long_matches(threshold, fill):
    streams = [pieces_stream(0xB1E + k) for k in range(150)]
    caps = []
    for k, s in enumerate(streams):
        st, data = oracle_decode("lz4", s, 1 << 22)
        assert st == libs.OK, f"the generator wrote an invalid stream ({k})"
        caps.append(len(data) - (1 if k % 6 == 5 else 0))
    streams += [last_literals(bytes(9))] * fill
    caps += [9] * fill
    print(f"[pieces] {len(streams)} chunks, threshold {threshold}", flush=True)
    with plan_by_threshold("lz4", threshold):
        res = check_against_oracle("lz4", "tuned", streams, caps)
    assert np.sum(res["status"][:150] != 0) == 25


@pytest.mark.parametrize("made", ["shaped", "slow_chunks", "chains"])
def test_edges_in_the_usual_windows(made, request):
    streams, caps, names = request.getfixturevalue(made)
    fill = 1100
    print(f"[queued edges] {made}: {len(streams)} chunks and {fill}", flush=True)
    with plan_by_threshold("lz4", 0):
        check_against_oracle("lz4", "tuned", streams + [last_literals(bytes(9))] * fill,
                             caps + [9] * fill, names + ["fill"] * fill)


@pytest.mark.parametrize("fmt", ["lz4", "snappy"])
@pytest.mark.parametrize("n", [2049, 5119, 5120, 5121, 5122, 10239, 10240, 10241])
def test_chunks_for_each_wave(fmt, n):
    rng = np.random.default_rng(n)
    codec = workload.CODEC_LZ4 if fmt == "lz4" else workload.CODEC_SNAPPY
    base = workload.build(codec, rng.integers(1, 600, 60), rng.integers(0, 3, 60),
                          rng.integers(1, 1 << 60, 60))
    which = rng.integers(0, 60, n)
    streams = [base.compressed(int(i)) for i in which]
    caps = [int(base.sizes[i]) for i in which]
    streams[3], caps[n - 2] = streams[3][:-1], 0
    print(f"[one wave] {fmt} {n} chunks", flush=True)
    with plan_by_threshold(fmt, 1 << 40):
        check_against_oracle(fmt, "tuned", streams, caps)


@pytest.mark.parametrize("fmt", ["lz4", "snappy"])
@pytest.mark.parametrize("threshold", [16 << 10, 1 << 40])
def test_every_cost_bin(fmt, threshold):
    codec = workload.CODEC_LZ4 if fmt == "lz4" else workload.CODEC_SNAPPY
    sizes = [int(1.18 ** k) for k in range(93)]  # 1 byte to 4 MiB, a few a bin
    b = workload.build(codec, sizes, [k % 3 for k in range(93)], range(1, 94))
    streams = [b.compressed(k) for k in range(93)] + [b.compressed(0), b"" if fmt == "lz4" else bytes(1)] + [b.compressed(20)] * 2400
    caps = sizes + [0, 0] + [sizes[20]] * 2400
    order = np.random.default_rng(4).permutation(len(streams))
    print(f"[cost bins] {fmt} {len(streams)} chunks, threshold {threshold}", flush=True)
    with plan_by_threshold(fmt, threshold):
        check_against_oracle(fmt, "tuned", [streams[i] for i in order], [caps[i] for i in order])
