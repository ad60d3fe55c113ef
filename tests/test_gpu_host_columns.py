"""Host columns of at most one chunk: the edges of the copy kernel's words, pieces and grid, columns
that a kernel cannot read (pageable or not on 8 bytes), and the rows around a chunk."""
import numpy as np
import pytest

from tpchq01_gpu_amd import q1

pytestmark = pytest.mark.gpu

CUTOFF = 729906


def _as_dicts(groups):
    return [vars(g) for g in groups]


def _columns(layout, rows):
    ref = q1.generate_host(q1.REFERENCE, 12, rows)
    cols = ref if layout == q1.REFERENCE else q1.generate_host(layout, 12, rows)
    return ref, cols


@pytest.mark.parametrize("layout", [q1.COMPRESSED, q1.UNCOMPRESSED, q1.REFERENCE])
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 33, 4096, 16_384, 16_385, 262_147, 2_700_001])
def test_one_chunk(ctx, oracle, layout, rows):
    ref, cols = _columns(layout, rows)
    want, _ = oracle.naive(ref, 0, rows, CUTOFF)
    pinned = ctx.pinned_columns(layout, rows)
    try:
        for name, v in pinned.items():
            v[:] = cols[name][:len(v)]
        for flags in (0, q1.LAUNCH_ASSUME_TPCH_DOMAIN):
            print("case", q1.LAYOUT_NAMES[layout], rows, flags, flush=True)
            launch = q1.make_launch(0, 0, 0, flags)
            for given in (pinned, cols):
                got = _as_dicts(ctx.run_streaming(layout, given, rows, CUTOFF, q1.AUTO, launch, 1 << 25, 2))
                assert got == want
                assert 0 < ctx.last_timing().kernel_ms <= ctx.last_timing().wall_ms
    finally:
        ctx.free_pinned_columns(pinned)


@pytest.mark.parametrize("placement", [q1.IN_REGISTERS, q1.PER_THREAD_SHARED_MEM, q1.GLOBAL])
def test_around_a_chunk(ctx, oracle, placement):
    """rows below, at and above chunk_rows, over one buffer; then columns that start one row into
    theirs, most of them not on 8 bytes."""
    chunk, layout = 65_536, q1.UNCOMPRESSED
    most = 2 * chunk + 77
    ref, cols = _columns(layout, most)
    pinned = ctx.pinned_columns(layout, most)
    try:
        for name, v in pinned.items():
            v[:] = cols[name][:len(v)]
        for rows in (0, chunk - 1, chunk, chunk + 1, most):
            want, _ = oracle.naive(ref, 0, rows, CUTOFF)
            print("case", placement, rows, flush=True)
            assert _as_dicts(ctx.run_streaming(layout, pinned, rows, CUTOFF, placement, None, chunk, 3)) == want
        want, _ = oracle.naive(ref, 1, 1 + 50_000, CUTOFF)
        shifted = {name: v[1:] for name, v in pinned.items()}
        assert _as_dicts(ctx.run_streaming(layout, shifted, 50_000, CUTOFF, placement, None, chunk, 3)) == want
    finally:
        ctx.free_pinned_columns(pinned)
