"""The batched kernel's request lists: searches of one, two and three looks, requests without
rows anywhere in the list, grids smaller than the list, and batches whose requests must share
fewer merge tables; every request equals q1_run of it alone, on calls in a row."""
import ctypes as C

import pytest

from tpchq01_gpu_amd import q1

pytestmark = pytest.mark.gpu

ROWS = 700_001


def _words(result):
    return bytes(result)


@pytest.fixture(scope="module")
def table(ctx):
    t = ctx.generate(q1.COMPRESSED, 11, ROWS)
    ranges = [(0, 1), (5, 0), (131, 4096), (0, ROWS), (77, 300_000), (ROWS, 0), (ROWS - 3, 3), (1000, 60_000)]
    alone = [_words(ctx.run_raw(t, b, n, 729950 + i, q1.AUTO)) for i, (b, n) in enumerate(ranges)]
    yield t, ranges, alone
    t.free()


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 129, 4096, 4097, 9000])
@pytest.mark.parametrize("shape", [(0, 0), (16, 0), (16, 7), (256, 300)])
def test_request_lists(ctx, table, n, shape):
    t, ranges, alone = table
    for start in (0, 1, 3):
        which = [(start + i * (1 if n < 200 else 5)) % len(ranges) for i in range(n)]
        reqs = (q1.Request * n)(*[q1.Request(t.handle, *ranges[k], 729950 + k, 0) for k in which])
        outs = (q1.Result * n)()
        launch = q1.make_launch(0, shape[0], shape[1])
        print("case", n, shape, start, flush=True)
        for _ in range(2):
            C.memset(outs, 0xEE, C.sizeof(outs))
            ctx.check(q1.lib.q1_run_batch(ctx.handle, reqs, n, C.byref(launch), outs), "q1_run_batch")
            wrong = [i for i in range(n) if _words(outs[i]) != alone[which[i]]]
            assert not wrong, (wrong[:5], len(wrong))


def test_requests_share_fewer_tables(ctx, table):
    """10,000 requests of 74 blocks each would take 80,000 tables, past the 65,536 kept."""
    t, ranges, alone = table
    n, k = 10_000, 4
    reqs = (q1.Request * n)(*[q1.Request(t.handle, *ranges[k], 729950 + k, 0)] * n)
    outs = (q1.Result * n)()
    launch = q1.make_launch(0, 16, 0)
    for _ in range(2):
        ctx.check(q1.lib.q1_run_batch(ctx.handle, reqs, n, C.byref(launch), outs), "q1_run_batch")
        assert all(_words(outs[i]) == alone[k] for i in range(n))


def test_no_request_has_rows(ctx, table):
    t = table[0]
    reqs = (q1.Request * 3)(*[q1.Request(t.handle, 10, 0, 729999, 0)] * 3)
    outs = (q1.Result * 3)()
    C.memset(outs, 0xEE, C.sizeof(outs))
    ctx.check(q1.lib.q1_run_batch(ctx.handle, reqs, 3, None, outs), "q1_run_batch")
    assert all(_words(o) == bytes(C.sizeof(q1.Result)) for o in outs)
