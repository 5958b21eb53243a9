"""Queued launches of little more than a block for each chunk: every block of
the pipelined kernel starts with a queue position of its own and draws the
next ones, so all are taken once, on both sides of the resident blocks (1024 on
256 CUs) and of two chunks a block, through every entry, against the plain
form: statuses, sizes and bytes."""
import pytest

import cudec_amd
from cudec_amd import workload
from cudec_amd.device import DeviceBatch
from tests.gpu_util import gpu
from tests.test_gpu_queued_launches import (POISON, arguments, check, clear, noalloc,
                                            plan_by_threshold, snapshot)

pytestmark = gpu

COUNTS = (1023, 1024, 1025, 1026, 1151, 2047, 2048, 2049)


@pytest.mark.parametrize("fmt", ["lz4", "snappy"])
@pytest.mark.parametrize("n", COUNTS)
def test_every_position_once(fmt, n):
    codec = workload.CODEC_LZ4 if fmt == "lz4" else workload.CODEC_SNAPPY
    b = workload.uneven(n, seed=n, codec=codec, min_size=512, octaves=7)
    comp = [b.compressed(i) for i in range(n)]
    for i in range(3, n, 17):
        comp[i] = comp[i][:-1]
    db = DeviceBatch.from_streams(comp, [int(s) for s in b.sizes], poison=POISON)
    db.reset_results()
    assert db.run(fmt, "plain") == 0
    want = snapshot(db)
    for threshold in (0, 16 << 10, 96 << 10):
        with plan_by_threshold(fmt, threshold):
            print(f"[positions] {fmt} {n} chunks, threshold {threshold}", flush=True)
            clear(db)
            assert db.run(fmt, "tuned") == 0
            check(db, want, "batch")
            clear(db)
            assert cudec_amd.lib().cudec_mi355x_parse_batch(cudec_amd.FORMAT_CODE[fmt],
                                                            *arguments(db), None) == 0
            assert (snapshot(db)[0] == want[0]).all()
            if fmt == "lz4":
                clear(db)
                assert noalloc(db) == 0
                check(db, want, "allocation-free")
