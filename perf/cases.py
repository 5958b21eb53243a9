"""The measured cases: the calls a program makes of this library, over their real range.

A case is one call of a public entry point:

* path "batch": the device batch entries (LZ4 and Snappy blocks, Zstandard
  frames), with compressed chunks and tables resident on the GPU, as a
  column store, a page cache or a request server calls them. `chunks`
  chunks, sizes log-uniform over [min, max] bytes (all `min` where the two
  are equal), odd sizes included. kinds "tokens" is the seeded token process
  (text-like, matches at offsets up to 64 KiB, many short overlapping ones);
  "mixed" is 80% of it, 10% incompressible and 10% highly repetitive chunks.
* path "frame": cudec_lz4f_decompress, one LZ4 frame from host memory to
  host memory, blocks of 64 KiB to 4 MiB, with a content checksum (the lz4
  tool's default) and, by option, block checksums.
* path "stream": cudec_lz4_decompress_stream_ctx, host chunks to host
  buffers through a kept streaming context.

A batch larger than DISTINCT bytes repeats its first DISTINCT bytes of
chunks at other addresses, so that inputs are made quickly; the device sees
different memory for every chunk.

Every output is whole bytes, so results are compared for equality.
"""
import math
import random
import struct

import numpy as np
import torch

import cudec_amd
from cudec_amd import workload

KIB, MIB = 1 << 10, 1 << 20
# Bytes of distinct chunk content made for one batch.
DISTINCT = 160 * MIB
CODECS = {"lz4": workload.CODEC_LZ4, "snappy": workload.CODEC_SNAPPY, "zstd": workload.CODEC_ZSTD}
ENTRIES = {"lz4": cudec_amd.cudec_lz4_decompress_batch,
           "snappy": cudec_amd.cudec_snappy_decompress_batch,
           "zstd": cudec_amd.cudec_zstd_decompress_batch}
# Compressed bytes per byte, (tokens, mixed), as the compressors give them for these workloads.
RATIO = {"lz4": (0.50, 0.58), "snappy": (0.50, 0.57), "zstd": (0.30, 0.35)}


def batch(fmt, chunks, lo, hi, kinds):
    return {"path": "batch", "format": fmt, "chunks": chunks, "min": lo, "max": hi, "kinds": kinds}


def listed():
    return [
        # One page read on its own: launch and queue latency.
        dict(batch("lz4", 1, 4 * KIB, 4 * KIB, "tokens"), name="lz4_page"),
        # A typical request of the serving loop: the geometric mean of its 1 to 256 chunks.
        dict(batch("lz4", 16, 4 * KIB, 1 * MIB, "tokens"), name="lz4_request"),
        # Rows or small pages of a table, in one call.
        dict(batch("lz4", 100003, 1 * KIB, 4 * KIB, "tokens"), name="lz4_records"),
        # Fixed 64 KiB blocks, the block size of most containers, 1 GiB of them.
        dict(batch("lz4", 16384, 64 * KIB, 64 * KIB, "tokens"), name="lz4_64k"),
        # A few large blocks of one file: the chip is mostly idle.
        dict(batch("lz4", 61, 1 * MIB, 4 * MIB, "mixed"), name="lz4_large"),
        # The benchmark's uneven batch: 1 KiB to 4 MiB, every kind of data.
        dict(batch("lz4", 20000, 1 * KIB, 4 * MIB, "mixed"), name="lz4_uneven"),
        # Snappy blocks of 64 KiB, the format's own fragment size, 512 MiB of them.
        dict(batch("snappy", 8192, 64 * KIB, 64 * KIB, "tokens"), name="snappy_64k"),
        # The uneven batch in Snappy.
        dict(batch("snappy", 10000, 1 * KIB, 4 * MIB, "mixed"), name="snappy_uneven"),
        # Zstandard frames of 64 KiB, 512 MiB of them.
        dict(batch("zstd", 8192, 64 * KIB, 64 * KIB, "tokens"), name="zstd_64k"),
        # The uneven batch as Zstandard frames; the large ones hold many blocks.
        dict(batch("zstd", 2000, 1 * KIB, 4 * MIB, "mixed"), name="zstd_uneven"),
        # A .lz4 file of ordinary size, read whole, with block checksums.
        {"name": "lz4_frame", "path": "frame", "bytes": 40 * MIB + 12345, "block": 256 * KIB,
         "block_sums": True, "kinds": "tokens"},
        # Host chunks in, host buffers out, through a kept context.
        {"name": "lz4_stream", "path": "stream", "chunks": 2048, "min": 16 * KIB,
         "max": 256 * KIB, "kinds": "tokens"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more call of the same ranges."""
    path = rng.choice(("lz4", "lz4", "lz4", "lz4", "snappy", "snappy", "zstd", "zstd", "frame",
                       "stream"))
    if path == "frame":
        return {"path": "frame", "bytes": _log(rng, 64 * KIB, 64 * MIB),
                "block": rng.choice((64 * KIB, 256 * KIB, MIB, 4 * MIB)),
                "block_sums": rng.random() < 0.5, "kinds": rng.choice(("tokens", "mixed"))}
    lo = _log(rng, 1 * KIB, 512 * KIB)
    hi = lo if rng.random() < 0.25 else min(4 * MIB, _log(rng, lo, 4 * MIB))
    # as many chunks as keep the call under the largest listed one's bytes
    most = {"lz4": 4096 * MIB, "snappy": 2048 * MIB, "zstd": 512 * MIB, "stream": 192 * MIB}[path]
    chunks = _log(rng, 1, min(120000, max(2, most // hi)))
    kinds = rng.choice(("tokens", "mixed"))
    if path == "stream":
        return {"path": "stream", "chunks": chunks, "min": lo, "max": hi, "kinds": kinds}
    return batch(path, chunks, lo, hi, kinds)


def _mean_size(lo, hi):
    return lo if lo == hi else (hi - lo) / math.log(hi / lo)


def work(case):
    """The compressed bytes read once and the decoded bytes written once."""
    mixed = case["kinds"] == "mixed"
    if case["path"] == "frame":
        n, fmt = case["bytes"], "lz4"
    else:
        n, fmt = case["chunks"] * _mean_size(case["min"], case["max"]), case.get("format", "lz4")
    return {"bytes": n * (1 + RATIO[fmt][mixed]), "flops": 0}


def exact(case, seed):
    """Outputs are bytes and whole numbers, with no computed floating value."""
    return None


def _chunks(case, codec, seed):
    """(distinct compressed batch, chunks of the whole batch / distinct ones)"""
    rng = np.random.default_rng(seed)
    lo, hi, n = case["min"], case["max"], case["chunks"]
    distinct = max(1, min(n, int(DISTINCT / _mean_size(lo, hi))))
    if lo == hi:
        sizes = np.full(distinct, lo, dtype=np.uint64)
    else:
        # one size from each of `distinct` equal slices of the logarithm, in an order that
        # the case decides, so that its outputs have the same shape for every seed
        own = np.random.default_rng([lo, hi, n])
        u = (np.arange(distinct) + own.random(distinct)) / distinct
        sizes = np.floor(lo * (hi / lo) ** own.permutation(u)).astype(np.uint64)
    kinds = np.zeros(distinct, dtype=np.int32)
    if case["kinds"] == "mixed":
        kinds = rng.choice(np.array([workload.KIND_TOKENS, workload.KIND_RANDOM,
                                     workload.KIND_REPETITIVE], dtype=np.int32),
                           size=distinct, p=[0.8, 0.1, 0.1])
    seeds = rng.integers(1, 1 << 62, size=distinct, dtype=np.uint64)
    return workload.build(codec, sizes, kinds, seeds)


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int64)).cuda()


def _prepare_batch(case, seed):
    b = _chunks(case, CODECS[case["format"]], seed)
    n = case["chunks"]
    which = np.arange(n) % b.n            # the distinct chunk that chunk i holds
    turn = (np.arange(n) // b.n).astype(np.uint64)
    comp = torch.from_numpy(b.comp).cuda()
    comp = comp.repeat(-(-n // b.n))
    sizes = b.sizes[which]
    out = torch.empty(int(sizes.sum()), dtype=torch.uint8, device="cuda")
    src = np.uint64(comp.data_ptr()) + turn * np.uint64(b.comp.size) + b.comp_off[which]
    dst = np.uint64(out.data_ptr()) + workload.offsets_of(sizes)
    return {"entry": ENTRIES[case["format"]], "n": n, "comp": comp, "out": out, "src": _dev(src),
            "src_sizes": _dev(b.comp_size[which]), "dst": _dev(dst), "caps": _dev(sizes),
            "results": torch.empty((n, 2), dtype=torch.int64, device="cuda")}


def _run_batch(s):
    st = s["entry"](s["src"].data_ptr(), s["src_sizes"].data_ptr(), s["dst"].data_ptr(),
                    s["caps"].data_ptr(), s["n"], s["results"].data_ptr(),
                    torch.cuda.current_stream().cuda_stream)
    if st != cudec_amd.CUDEC_OK:
        raise RuntimeError(f"batch call refused: {st}")
    return {"out": s["out"], "results": s["results"]}


def _xxh32(arrays):
    """XXH32 (seed 0) of each of the arrays, on the GPU."""
    data = torch.from_numpy(np.concatenate(arrays)).cuda()
    sizes = np.array([a.size for a in arrays], dtype=np.uint64)
    ptrs, lens = _dev(np.uint64(data.data_ptr()) + workload.offsets_of(sizes)), _dev(sizes)
    sums = torch.empty(len(arrays), dtype=torch.int32, device="cuda")
    st = cudec_amd.lib().cudec_mi355x_xxh32_batch(ptrs.data_ptr(), lens.data_ptr(), len(arrays), 0,
                                                  sums.data_ptr(),
                                                  torch.cuda.current_stream().cuda_stream)
    if st != cudec_amd.CUDEC_OK:
        raise RuntimeError(f"checksum call refused: {st}")
    return sums.cpu().numpy().view(np.uint32)


def _prepare_frame(case, seed):
    rng = random.Random(seed)
    left, block, sizes = case["bytes"], case["block"], []
    while left:
        sizes.append(min(left, block))
        left -= sizes[-1]
    kinds = [0 if case["kinds"] == "tokens" else rng.choices((0, 1, 2), (8, 1, 1))[0]
             for _ in sizes]
    b = workload.build(workload.CODEC_LZ4, sizes, kinds, [rng.randrange(1, 1 << 62) for _ in sizes])
    code = {64 * KIB: 4, 256 * KIB: 5, MIB: 6, 4 * MIB: 7}[block]
    # version 01, independent blocks, content checksum, block checksums by option
    head = bytes((0x64 | (0x10 if case["block_sums"] else 0), code << 4))
    stored, parts = [], []
    for i in range(b.n):
        o, n = int(b.comp_off[i]), int(b.comp_size[i])
        if n < sizes[i]:
            parts.append(b.comp[o:o + n])
        else:
            o = int(b.orig_off[i])
            parts.append(b.orig[o:o + sizes[i]])
        stored.append(n >= sizes[i])
    sums = _xxh32([np.frombuffer(head, np.uint8).copy(), b.orig] + parts)
    frame = [struct.pack("<I", 0x184D2204), head, bytes(((int(sums[0]) >> 8) & 255,))]
    for i, p in enumerate(parts):
        frame.append(struct.pack("<I", p.size | (0x80000000 if stored[i] else 0)))
        frame.append(p.tobytes())
        if case["block_sums"]:
            frame.append(struct.pack("<I", int(sums[2 + i])))
    frame += [struct.pack("<I", 0), struct.pack("<I", int(sums[1]))]
    return {"frame": b"".join(frame), "capacity": case["bytes"]}


def _run_frame(s):
    st, out = cudec_amd.cudec_lz4f_decompress(s["frame"], s["capacity"])
    if st != cudec_amd.CUDEC_OK:
        raise RuntimeError(f"frame call refused: {st}")
    return np.frombuffer(out, dtype=np.uint8)


class _Context:
    """A streaming context that lives as long as the state that holds it."""

    def __init__(self):
        st, self.handle = cudec_amd.cudec_stream_ctx_create()
        if st != cudec_amd.CUDEC_OK:
            raise RuntimeError(f"no streaming context: {st}")

    def __del__(self):
        cudec_amd.cudec_stream_ctx_destroy(self.handle)


def _prepare_stream(case, seed):
    b = _chunks(case, workload.CODEC_LZ4, seed)
    n = case["chunks"]
    which = np.arange(n) % b.n
    sizes = np.ascontiguousarray(b.sizes[which])
    out = np.zeros(int(sizes.sum()), dtype=np.uint8)
    return {"ctx": _Context(), "n": n, "comp": b.comp, "out": out,
            "src": np.uint64(b.comp.ctypes.data) + b.comp_off[which],
            "src_sizes": np.ascontiguousarray(b.comp_size[which]),
            "dst": np.uint64(out.ctypes.data) + workload.offsets_of(sizes), "caps": sizes,
            "results": np.zeros((n, 2), dtype=np.int64)}


def _run_stream(s):
    st = cudec_amd.cudec_lz4_decompress_stream_ctx(
        s["ctx"].handle, s["src"].ctypes.data, s["src_sizes"].ctypes.data, s["dst"].ctypes.data,
        s["caps"].ctypes.data, s["n"], cudec_amd.CUDEC_MEM_HOST, s["results"].ctypes.data)
    if st != cudec_amd.CUDEC_OK:
        raise RuntimeError(f"stream call refused: {st}")
    return {"out": s["out"], "results": s["results"]}


def prepare(case, seed):
    make = {"batch": _prepare_batch, "frame": _prepare_frame, "stream": _prepare_stream}
    return dict(make[case["path"]](case, seed), path=case["path"])


def run(state):
    return {"batch": _run_batch, "frame": _run_frame, "stream": _run_stream}[state["path"]](state)
