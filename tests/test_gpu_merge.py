"""The merge at the end of a scan kernel: grids of one block, around the 8 blocks up to which
q1_run's blocks each leave a record for the host, around the 64 tables of a merge set, around
the 144 blocks from which q1_enqueue merges through a set, and of many blocks per table; twice
in a row, since every launch must leave its set zero."""
import ctypes as C

import numpy as np
import pytest

from tpchq01_gpu_amd import q1

pytestmark = pytest.mark.gpu

BLOCKS = [1, 2, 8, 9, 17, 63, 64, 65, 129, 143, 144, 1000]
LANES, LANE_ROWS = 64, 16


def _as_dicts(groups):
    return [vars(g) for g in groups]


def _columns(layout, rows, wide):
    """Rows of the generator; wide: with discounts above 100 and prices near 2^32 (and, in
    the reference layout, 2^40), so that sums turn negative and pass 2^64."""
    ref = q1.generate_host(q1.REFERENCE, 7, rows)
    if wide:
        ref["discount"][::3] = 200
        ref["extended_price"][::2] = 4_000_000_000 if layout == q1.COMPRESSED else 1 << 40
    return ref, (q1.compress_columns(ref, rows) if layout == q1.COMPRESSED else ref)


@pytest.mark.parametrize("layout", [q1.COMPRESSED, q1.REFERENCE])
@pytest.mark.parametrize("wide", [False, True])
def test_grids_of_every_merge(ctx, oracle, layout, wide):
    import torch
    per = LANES * LANE_ROWS
    most = max(BLOCKS) * per
    ref, cols = _columns(layout, most, wide)
    t = ctx.upload(layout, cols, most)
    sums = torch.zeros(48, dtype=torch.int64, device="cuda")
    own = torch.cuda.Stream()
    for blocks in BLOCKS:
        rows = blocks * per - 5
        want, _ = oracle.naive(ref, 0, rows, 729999)
        for placement in (q1.PER_THREAD_SHARED_MEM, q1.IN_REGISTERS, q1.GLOBAL):
            launch = q1.make_launch(LANES, LANE_ROWS, 0, 0 if wide else q1.LAUNCH_ASSUME_TPCH_DOMAIN)
            for again in range(2):
                print("case", q1.LAYOUT_NAMES[layout], "wide", wide, blocks, placement, again, flush=True)
                assert _as_dicts(ctx.run(t, 0, rows, 729999, placement, launch)) == want
                assert ctx.last_timing().num_blocks == blocks
            if placement == q1.GLOBAL:
                continue
            dev = t.device_columns()
            for stream in (None, own.cuda_stream):
                torch.cuda.synchronize()
                sums.zero_()
                torch.cuda.synchronize()
                for _ in range(3):
                    ctx.check(q1.lib.q1_enqueue(ctx.handle, placement, layout, C.byref(launch), sums.data_ptr(),
                                                C.byref(dev), 0, rows, 729999, stream), "q1_enqueue")
                torch.cuda.synchronize()
                got = q1.DeviceAggregates.from_buffer_copy(np.ascontiguousarray(sums.cpu().numpy()).tobytes())
                r = q1.Result()
                q1.lib.q1_aggregates_to_result(C.byref(got), C.byref(r))
                assert _as_dicts(q1.result_to_list(r)) == [{k: 3 * v for k, v in g.items()} for g in want]
    t.free()


def test_more_launches_in_flight_than_merge_sets(ctx, oracle):
    """1,200 launches enqueued at once on four streams, more than the 256 merge sets: the ones
    without a set merge directly, and the next ones find their sets zero."""
    import torch
    rows, chunk = 400_000, 200_000
    ref, cols = _columns(q1.COMPRESSED, rows, False)
    want, _ = oracle.naive(ref, 0, rows, 729999)
    t = ctx.upload(q1.COMPRESSED, cols, rows)
    dev = t.device_columns()
    launch = q1.make_launch(LANES, LANE_ROWS, 0, q1.LAUNCH_ASSUME_TPCH_DOMAIN)   # 196 blocks each
    streams = [torch.cuda.Stream() for _ in range(4)]
    for turn in range(2):
        sums = [torch.zeros(48, dtype=torch.int64, device="cuda") for _ in streams]
        busy = torch.zeros(1 << 28, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        for s in streams:       # the launches queue up behind these
            with torch.cuda.stream(s):
                for _ in range(20):
                    busy.add_(1)
        for i in range(300):
            for s, out in zip(streams, sums):
                ctx.check(q1.lib.q1_enqueue(ctx.handle, q1.PER_THREAD_SHARED_MEM, q1.COMPRESSED, C.byref(launch),
                                            out.data_ptr(), C.byref(dev), chunk * (i % 2), chunk, 729999,
                                            s.cuda_stream), "q1_enqueue")
        torch.cuda.synchronize()
        for out in sums:
            got = q1.DeviceAggregates.from_buffer_copy(np.ascontiguousarray(out.cpu().numpy()).tobytes())
            r = q1.Result()
            q1.lib.q1_aggregates_to_result(C.byref(got), C.byref(r))
            assert _as_dicts(q1.result_to_list(r)) == [{k: 150 * v for k, v in g.items()} for g in want]
    t.free()
