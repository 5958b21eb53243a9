"""The host-memory entries where their staging changes shape: streaming calls
of one wave, of as many waves as there are slots and of more, with several
copying threads, to host and device outputs, with chunks that fail; and
frames whose blocks go up in one run or several."""
import ctypes
import struct

import numpy as np
import pytest

import cudec_amd
from cudec_amd import workload
from tests import libs
from tests.gpu_util import POISON, gpu

pytestmark = gpu

RES = np.dtype([("status", "<i4"), ("reserved", "<u4"), ("bytes_written", "<u8")])


@pytest.fixture(scope="module")
def chunks():
    sizes = [1, 70, 5000, 65536, 300001, 1 << 20, 900_017]
    return workload.build(workload.CODEC_LZ4, sizes, [0, 1, 2, 0, 2, 0, 0], range(1, 8))


@pytest.mark.parametrize("space", ["host", "device"])
@pytest.mark.parametrize("n", [5, 61, 140, 503])  # about 2, 30, 70 and 250 MB
def test_stream_waves(chunks, n, space):
    import torch
    b = chunks
    which = np.arange(n) * 3 % b.n
    sizes = b.sizes[which].astype(np.uint64)
    comp = np.ascontiguousarray(b.comp)
    src = np.uint64(comp.ctypes.data) + b.comp_off[which].astype(np.uint64)
    src_sizes = b.comp_size[which].astype(np.uint64)
    caps = sizes.copy()
    bad = {2: "short", n - 1: "room"}
    caps[2] -= 1
    caps[n - 1] += 13
    offs = workload.offsets_of(caps)
    total = int(caps.sum())
    if space == "host":
        out = np.full(total, POISON, dtype=np.uint8)
        base, mem = out.ctypes.data, cudec_amd.CUDEC_MEM_HOST
    else:
        dev = torch.full((total,), POISON, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        base, mem = dev.data_ptr(), cudec_amd.CUDEC_MEM_DEVICE
    dst = np.uint64(base) + offs.astype(np.uint64)
    st, ctx = cudec_amd.cudec_stream_ctx_create()
    assert st == 0
    try:
        for turn in range(2):  # a new context, and one with its staging
            res = np.zeros(n, dtype=RES)
            st = cudec_amd.cudec_lz4_decompress_stream_ctx(
                ctx, src.ctypes.data, src_sizes.ctypes.data, dst.ctypes.data, caps.ctypes.data, n,
                mem, res.ctypes.data)
            assert st == libs.TOO_SMALL
            got = out if space == "host" else dev.cpu().numpy()
            for i in range(n):
                if bad.get(i) == "short":
                    assert res["status"][i] == libs.TOO_SMALL and res["bytes_written"][i] == 0
                    continue
                assert res["status"][i] == 0 and res["bytes_written"][i] == sizes[i], i
                o, s = int(offs[i]), int(sizes[i])
                assert np.array_equal(got[o:o + s], np.frombuffer(b.original(int(which[i])),
                                                                  np.uint8)), i
                assert np.all(got[o + s:o + int(caps[i])] == POISON), i
    finally:
        cudec_amd.cudec_stream_ctx_destroy(ctx)


@pytest.mark.parametrize("sums", [False, True])
@pytest.mark.parametrize("stored", ["none", "all", "some", "first", "long"])
def test_frame_runs(chunks, stored, sums):
    """Stored blocks are left out of the upload (unless their checksums are
    checked); short ones are crossed, longer ones end a run."""
    b = chunks
    order = [2, 3, 4, 2, 5, 1, 6, 3, 3, 2, 1, 5] * 3
    head = bytes((0x60 | (0x10 if sums else 0), 7 << 4))
    frame = struct.pack("<I", 0x184D2204) + head
    frame += bytes(((_xxh32(head) >> 8) & 255,))
    want = []
    for i, c in enumerate(order):
        plain, comp = bytes(b.original(c)), bytes(b.compressed(c))
        raw = {"none": False, "all": True, "some": i % 3 == 1, "first": i < 4,
               "long": len(plain) > 100_000}[stored]
        body = plain if raw else comp
        frame += struct.pack("<I", len(body) | (0x80000000 if raw else 0)) + body
        if sums:
            frame += struct.pack("<I", _xxh32(body))
        want.append(plain)
    frame += struct.pack("<I", 0)
    want = b"".join(want)
    st, out = cudec_amd.cudec_lz4f_decompress(frame, len(want))
    assert st == 0 and out == want
    st, out = cudec_amd.cudec_lz4f_decompress(frame, len(want) + 5)
    assert st == 0 and out == want
    assert cudec_amd.cudec_lz4f_decompress(frame, len(want) - 1) == (libs.TOO_SMALL, b"")


def _xxh32(data):
    import torch
    d = torch.from_numpy(np.frombuffer(data, np.uint8).copy()).cuda()
    ptr = torch.tensor([d.data_ptr()], dtype=torch.int64, device="cuda")
    size = torch.tensor([len(data)], dtype=torch.int64, device="cuda")
    sums = torch.zeros(1, dtype=torch.int32, device="cuda")
    assert cudec_amd.lib().cudec_mi355x_xxh32_batch(
        ctypes.c_void_p(ptr.data_ptr()), ctypes.c_void_p(size.data_ptr()), 1, 0,
        ctypes.c_void_p(sums.data_ptr()),
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    return int(sums.cpu().numpy().view(np.uint32)[0])
