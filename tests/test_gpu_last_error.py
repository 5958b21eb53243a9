"""A failed call reports its failure in its status alone: the GPU call that the
program makes next, torch's here, does not report it again."""
import numpy as np
import torch

import cudec_amd
from tests import libs
from tests.gpu_util import gpu

pytestmark = gpu


def test_streaming_call_without_memory():
    src, out = np.zeros(1, np.uint8), np.zeros(1, np.uint8)
    ptrs = [np.array([a.ctypes.data], np.uint64) for a in (src, out)]
    size, cap = np.array([1], np.uint64), np.array([1 << 60], np.uint64)
    res = np.zeros((1, 2), np.int64)
    st, ctx = cudec_amd.cudec_stream_ctx_create()
    assert st == libs.OK
    print("[last error] staging of 2^60 bytes", flush=True)
    st = cudec_amd.cudec_lz4_decompress_stream_ctx(
        ctx, ptrs[0].ctypes.data, size.ctypes.data, ptrs[1].ctypes.data, cap.ctypes.data, 1,
        cudec_amd.CUDEC_MEM_HOST, res.ctypes.data)
    assert st == libs.DEVICE
    assert torch.cat([torch.zeros(3, device="cuda"), torch.ones(3, device="cuda")]).sum() == 3
    cudec_amd.cudec_stream_ctx_destroy(ctx)
