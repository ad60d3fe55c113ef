"""The any-value kernel at the limits of its LDS words: every field driven to the smallest and
largest value of its column type, for as many rows per lane as the kernel takes, in every
launch width; and tuples_per_thread beyond that, which become more blocks."""
import numpy as np
import pytest

from tpchq01_gpu_amd import q1

pytestmark = pytest.mark.gpu

# extreme values per layout and column
EXTREMES = {
    q1.COMPRESSED: dict(quantity=(0, 255), extended_price=(0, 2**32 - 1), discount=(0, 255), tax=(0, 255)),
    q1.UNCOMPRESSED: dict(quantity=(-2**31, 2**31 - 1), extended_price=(-2**63, 2**63 - 1), discount=(-128, 127),
                          tax=(-128, 127)),
    q1.REFERENCE: dict(quantity=(-2**63, 2**63 - 1), extended_price=(-2**63, 2**63 - 1),
                       discount=(-2**63, 2**63 - 1), tax=(-2**63, 2**63 - 1)),
}


def _as_dicts(groups):
    return [vars(g) for g in groups]


def _case(layout, rows, choice, rng):
    """Device columns whose values all take extreme `choice` (per column, or at random when
    None), and the same rows as the oracle's reference columns."""
    cols = q1.generate_host(layout, 3, rows)
    for name, (lo, hi) in EXTREMES[layout].items():
        if choice is None:
            v = np.where(rng.integers(0, 2, rows) == 0, np.array(lo, cols[name].dtype), np.array(hi, cols[name].dtype))
        else:
            v = np.full(rows, (lo, hi)[choice[name]], cols[name].dtype)
        cols[name][:rows] = v
    ref = q1.generate_host(q1.REFERENCE, 3, rows)
    for name in EXTREMES[layout]:
        ref[name] = cols[name].astype(np.int64)
    if layout == q1.COMPRESSED:
        ref["quantity"] *= 100
    return cols, ref


@pytest.mark.parametrize("layout", [q1.COMPRESSED, q1.UNCOMPRESSED, q1.REFERENCE])
def test_every_field_at_its_limits(ctx, oracle, layout):
    rng = np.random.default_rng(8)
    rows = 4 * 64 * 256 + 3 * 64 * 256 + 77
    names = list(EXTREMES[layout])
    choices = [{n: (k >> i) & 1 for i, n in enumerate(names)} for k in range(16)] + [None, None]
    for choice in choices:
        cols, ref = _case(layout, rows, choice, rng)
        want, _ = oracle.naive(ref, 0, rows, 730100)
        t = ctx.upload(layout, cols, rows)
        for shape in ((64, 256), (128, 128), (256, 256), (256, 1024), (64, 272), (64, 16384), (0, 0)):
            print("case", q1.LAYOUT_NAMES[layout], choice, shape, flush=True)
            got = _as_dicts(ctx.run(t, 0, rows, 730100, q1.PER_THREAD_SHARED_MEM, q1.make_launch(*shape)))
            assert got == want, (choice, shape)
        lanes = 128 if layout == q1.COMPRESSED else 256
        assert ctx.last_timing().tuples_per_thread <= lanes
        t.free()


@pytest.mark.parametrize("layout", [q1.COMPRESSED, q1.UNCOMPRESSED, q1.REFERENCE])
def test_one_group_only(ctx, oracle, layout):
    """All rows in one group, so that its sums grow as fast as they can, over more blocks than
    a merge set has tables; a range that starts and ends inside tiles."""
    rows = 1_300_021
    cols, ref = _case(layout, rows, {n: 1 for n in EXTREMES[layout]}, None)
    cols["return_flag"][:] = 0 if layout == q1.COMPRESSED else ord("A")
    cols["line_status"][:] = 0 if layout == q1.COMPRESSED else ord("F")
    ref["return_flag"][:], ref["line_status"][:] = ord("A"), ord("F")
    t = ctx.upload(layout, cols, rows)
    for begin, end in ((0, rows), (77, rows - 13), (131, 132)):
        want, _ = oracle.naive(ref, begin, end, 730100)
        for shape in ((64, 16), (128, 128), (0, 0)):
            print("case", q1.LAYOUT_NAMES[layout], begin, end, shape, flush=True)
            got = _as_dicts(ctx.run(t, begin, end - begin, 730100, q1.IN_REGISTERS, q1.make_launch(*shape)))
            assert got == want
    t.free()


@pytest.mark.parametrize("layout", [q1.COMPRESSED, q1.REFERENCE])
def test_grids_a_caller_chooses(ctx, layout):
    """num_blocks is held against the caller's tuples_per_thread, or the shape taken for 0, as
    before: large enough runs, too small is refused."""
    rows = 500_000
    cols, _ = _case(layout, rows, None, np.random.default_rng(1))
    t = ctx.upload(layout, cols, rows)
    whole = ctx.run(t)
    for tpb, tpt in ((256, 1024), (64, 16384), (128, 512)):
        least = -(-rows // (tpb * tpt))
        assert ctx.run(t, launch=q1.make_launch(tpb, tpt, least)) == whole
        assert ctx.run(t, launch=q1.make_launch(tpb, tpt, least + 100)) == whole
        if least > 1:
            with pytest.raises(q1.Q1Error):
                ctx.run(t, launch=q1.make_launch(tpb, tpt, least - 1))
    t.free()


@pytest.mark.parametrize("layout,fit,most", [(q1.COMPRESSED, 1024, 1024), (q1.UNCOMPRESSED, 640, 512),
                                             (q1.REFERENCE, 384, 256)])
def test_default_rows_per_lane(ctx, oracle, layout, fit, most):
    """The rows at which the default shape changes: 16 per lane up to `fit` lanes per compute
    unit, one round of `most` lanes up to 128 rows each, then rounds of short blocks."""
    units = 256
    edges = [16 * units * fit, 2 * 16 * units * most, 128 * units * most]
    rows = edges[-1] + 1
    cols, ref = _case(layout, rows, None, np.random.default_rng(9))
    t = ctx.upload(layout, cols, rows)
    for n in sorted({e + d for e in edges for d in (0, 1)}):
        print("case", q1.LAYOUT_NAMES[layout], n, flush=True)
        want, _ = oracle.naive(ref, 0, n, 730100)
        assert _as_dicts(ctx.run(t, 0, n, 730100)) == want, n
        lane = ctx.last_timing().tuples_per_thread
        assert lane == 16 if n <= edges[0] else 16 < lane <= 128
    t.free()
