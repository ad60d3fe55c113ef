"""The device's value-domain check (run by upload, wrap and refresh): one value outside the
TPC-H domain, in any column and at any place of it, sends a table to the any-value kernel."""
import ctypes as C

import numpy as np
import pytest

from tpchq01_gpu_amd import q1

pytestmark = pytest.mark.gpu

# the largest value inside the domain, per column
TOP = {"discount": 15, "tax": 15, "quantity": 63, "extended_price": (1 << 24) - 1}


def _columns(layout, rows):
    cols = q1.empty_columns(layout, rows)
    for name, top in TOP.items():
        cols[name][:] = top * 100 if name == "quantity" and layout != q1.COMPRESSED else top
    return cols


def _ran_any_value(ctx, table):
    ctx.run(table, 0, 1, 729999, q1.PER_THREAD_SHARED_MEM)
    return ctx.last_timing().placement != q1.PER_THREAD_SHARED_MEM


@pytest.mark.parametrize("layout", [q1.REFERENCE, q1.UNCOMPRESSED, q1.COMPRESSED])
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 31, 4099, 300_007, 9_000_001])
def test_one_value_outside_the_domain(ctx, layout, rows):
    cols = _columns(layout, rows)
    t = ctx.upload(layout, cols, rows)
    assert not _ran_any_value(ctx, t)          # every value at its limit: inside
    dev = t.device_columns()
    w = ctx.wrap(layout, dev, rows)
    places = sorted({0, rows // 2, max(rows - 17, 0), rows - 1, min(rows - 1, 4096 * 63 + 5)})
    for name in TOP:
        host = cols[name]
        outside = [int(host[0]) + 1]
        if host.dtype.kind == "i":
            outside.append(-1)
        if host.dtype.itemsize == 8:
            outside.append(1 << 32)
        for place in places:
            for value in outside:
                kept = host[place].copy()
                host[place] = value
                print("case", q1.LAYOUT_NAMES[layout], rows, name, place, value, flush=True)
                t2 = ctx.upload(layout, cols, rows) if rows < 10_000 else None
                if t2 is None:                 # a larger table: overwrite the value in place
                    at = getattr(dev, name) + place * host.itemsize
                    src = np.array([value], dtype=host.dtype)
                    _copy_to_device(at, src)
                    ctx.check(q1.lib.q1_table_refresh_domain(ctx.handle, w.handle), "refresh")
                    assert _ran_any_value(ctx, w)
                    host[place] = kept
                    _copy_to_device(at, host[place:place + 1])
                else:
                    assert _ran_any_value(ctx, t2)
                    t2.free()
                    host[place] = kept
    ctx.check(q1.lib.q1_table_refresh_domain(ctx.handle, w.handle), "refresh")
    assert not _ran_any_value(ctx, w)
    w.free()
    t.free()


def _copy_to_device(address, array):
    hip = C.CDLL(None)
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    assert hip.hipMemcpy(address, array.ctypes.data, array.nbytes, 1) == 0
