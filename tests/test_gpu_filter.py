"""Filter bitmaps built one after another: each takes the memory of the one freed before it when
that is large enough, also while a launch on another stream still reads it."""
import ctypes as C

import numpy as np
import pytest

from tpchq01_gpu_amd import q1

pytestmark = pytest.mark.gpu


def _as_dicts(groups):
    return [vars(g) for g in groups]


def _check(ctx, oracle, ref, table, rows, cutoff):
    f = ctx.build_filter(table, cutoff)
    want, _ = oracle.naive(ref, 0, rows, cutoff)
    assert _as_dicts(ctx.run(f, 0, rows, 0)) == want, (rows, cutoff)
    return f


def test_bitmaps_of_many_sizes(ctx, oracle):
    """Growing, shrinking and equal sizes, one and two alive at a time."""
    most = 300_007
    ref = q1.generate_host(q1.REFERENCE, 5, most)
    alive = None
    for i, rows in enumerate([1, 31, 32, 33, most, 4099, most, 65_536, 17, most - 31, most]):
        t = ctx.upload(q1.COMPRESSED, q1.compress_columns(ref, rows), rows)
        f = _check(ctx, oracle, ref, t, rows, 728_000 + 300 * i)
        if i % 3 == 0:
            if alive:
                alive.free()
            alive = f
        else:
            f.free()
        _check(ctx, oracle, ref, t, rows, 729_000 + 100 * i).free()
        t.free()
    if alive:
        alive.free()


def test_freed_while_another_stream_reads_it(ctx, oracle):
    import torch
    rows = 6_000_001
    ref = q1.generate_host(q1.REFERENCE, 6, rows)
    t = ctx.upload(q1.COMPRESSED, q1.compress_columns(ref, rows), rows)
    own = torch.cuda.Stream()
    sums = [torch.zeros(48, dtype=torch.int64, device="cuda") for _ in range(8)]
    torch.cuda.synchronize()
    cutoffs = [728_500 + 200 * i for i in range(len(sums))]
    for s, cutoff in zip(sums, cutoffs):
        f = ctx.build_filter(t, cutoff)
        cols = f.device_columns()
        ctx.check(q1.lib.q1_enqueue(ctx.handle, q1.IN_REGISTERS, q1.COMPRESSED_PUSHDOWN, None, C.c_void_p(s.data_ptr()),
                                    C.byref(cols), 0, rows, 0, C.c_void_p(own.cuda_stream)), "q1_enqueue")
        f.free()
    torch.cuda.synchronize()
    for s, cutoff in zip(sums, cutoffs):
        want, _ = oracle.naive(ref, 0, rows, cutoff)
        got = q1.DeviceAggregates.from_buffer_copy(np.ascontiguousarray(s.cpu().numpy()).tobytes())
        r = q1.Result()
        q1.lib.q1_aggregates_to_result(C.byref(got), C.byref(r))
        assert _as_dicts(q1.result_to_list(r)) == want, cutoff
    t.free()
