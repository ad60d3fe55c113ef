"""The calls whose speed is watched: Q1 as programs run it through the C ABI's Python binding,
over the whole range of table sizes, column layouts and ways of handing rows over.

The rows are TPC-H-like lineitem rows made on the GPU by torch from the seed (dates over
1992-1998, quantities 1..50, prices quantity x 900.00..2099.99, discounts 0..0.10, taxes
0..0.08); every entry point returns integers, so two runs agree to the last bit.  A result is
the 6 x 8 words of q1_result: quantity, price, disc_price (lo, hi), charge (lo, hi), discount
and count of every group.
"""
import ctypes
import functools
import math
import random

import numpy as np
import torch

from tpchq01_gpu_amd import q1, serving

CUTOFF_FIRST, CUTOFF_LAST = 729906, 730088  # 1998-06-01 .. 1998-11-30
FRAME = 727563                              # 1992-01-01, the zero of the compressed ship dates
LAYOUTS = {"reference": q1.REFERENCE, "uncompressed": q1.UNCOMPRESSED, "compressed": q1.COMPRESSED}
BITS = {"reference": 304, "uncompressed": 160, "compressed": 75}
RUN_PLACEMENTS = ["auto", "in_registers", "in_registers_per_thread", "local_mem", "global"]


def _case(way, layout, rows, begin=0, placement="auto", wide=False, requests=1, **more):
    return dict(way=way, layout=layout, rows=rows, begin=begin, placement=placement, wide=wide, requests=requests,
                **more)


def listed():
    return [
        # The shortest query: one small table, where the launches and the wait are the cost.
        _case("run", "compressed", 5_003, name="run_compressed_5k"),
        # A slice of the serving workload's smallest table, starting at an arbitrary row.
        _case("run", "compressed", 1_000_003, begin=77, name="run_compressed_1m_slice"),
        # The 6M-row sample of the CPU baselines with the Python binding's default placement.
        _case("run", "uncompressed", 6_000_000, placement="in_registers", name="run_uncompressed_6m_registers"),
        # The 60M-row uncompressed sample with the reference driver's default placement.
        _case("run", "uncompressed", 60_000_000, placement="in_registers_per_thread",
              name="run_uncompressed_60m_per_thread"),
        # The headline: 600M resident compressed rows, placement chosen by the tuning table.
        _case("run", "compressed", 600_000_000, name="run_compressed_600m"),
        # A table outside the TPC-H value domain: bulk orders, quantities up to 200.
        _case("run", "compressed", 60_000_007, wide=True, name="run_compressed_60m_bulk_orders"),
        # Columns that another program just wrote (torch tensors), wrapped and queried once.
        _case("wrap", "compressed", 60_000_000, name="wrap_and_run_compressed_60m"),
        # Filter pushdown rebuilt for each query's own cutoff: bitmap, query, release.
        _case("pushdown", "compressed", 60_000_000, name="pushdown_compressed_60m"),
        # The reference's own loop: kernel launches of 2,097,152 rows of plain columns, no
        # promise about their values, accumulating on the caller's stream.
        _case("enqueue", "reference", 60_000_000, chunk=2_097_152, name="enqueue_reference_60m_chunks"),
        # The batched workload: 256 tables of 10^4..2*10^7 rows in one launch.
        _case("batch", "compressed", 20_000_000, requests=256, name="batch_256_requests"),
        # A burst of arrivals at the server: 64 slices of 8 tables of 1M..60M rows.
        _case("serve", "compressed", 60_000_000, requests=64, name="serve_burst_64"),
        # The reference driver's default mode: rows in pinned host memory, streamed.
        _case("stream", "compressed", 60_000_000, name="stream_host_60m"),
    ]


def _log_uniform(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng: random.Random):
    way = rng.choice(["run", "run", "run", "wrap", "pushdown", "enqueue", "batch", "serve", "stream"])
    layout = rng.choice(["compressed", "compressed", "uncompressed", "reference"])
    if way in ("pushdown", "batch", "serve", "stream"):
        layout = "compressed"
    most = {"run": 400_000_000, "wrap": 100_000_000, "pushdown": 200_000_000, "enqueue": 100_000_000,
            "batch": 10_000_000, "serve": 40_000_000, "stream": 60_000_000}[way]
    rows = _log_uniform(rng, 5_000, most * 75 // BITS[layout])
    if way == "run":
        return _case(way, layout, rows, begin=rng.choice([0, rng.randrange(1, 1000)]),
                     placement=rng.choice(["auto", "auto"] + RUN_PLACEMENTS), wide=rng.random() < 0.2)
    if way == "enqueue":
        return _case(way, layout, rows, chunk=_log_uniform(rng, 200_000, 40_000_000) // 32 * 32)
    if way in ("batch", "serve"):
        rows = _log_uniform(rng, 100_000, most)
        return _case(way, layout, rows, requests=rng.randrange(2, 150))
    return _case(way, layout, rows, wide=way == "wrap" and rng.random() < 0.2)


# --- the rows ----------------------------------------------------------------------------
def _plain_rows(rows, seed, wide):
    """Chunks of rows as plain integer columns: (first row, {name: int tensor})."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def draw_int(lo, hi, n, dtype=torch.int32):
        return torch.randint(lo, hi, (n,), generator=g, device="cuda", dtype=dtype)

    step = 1 << 26
    for r0 in range(0, rows, step):
        n = min(step, rows - r0)
        ship = draw_int(727564, 727564 + 2526, n)
        late = ship + draw_int(1, 31, n) > 728826
        rf = torch.where(late, 1, 2 * draw_int(0, 2, n))   # N, else A or R
        ls = (ship > 728826).to(torch.int32)               # F or O
        qty = draw_int(1, 201 if wide else 51, n)
        price = qty * draw_int(90_000, 210_000, n)
        yield r0, dict(ship=ship, rf=rf, ls=ls, qty=qty, price=price, disc=draw_int(0, 11, n, torch.int8),
                       tax=draw_int(0, 9, n, torch.int8))


def _packed(codes, bits):
    """Codes of `bits` bits, least significant first, in 32-bit words."""
    per = 32 // bits
    pad = torch.nn.functional.pad(codes.to(torch.int32), (0, -len(codes) % per)).view(-1, per)
    out = torch.zeros(len(pad), dtype=torch.int32, device=codes.device)
    for j in range(per):
        out |= pad[:, j] << (bits * j)
    return out


def _as_layout(layout, p):
    if layout == "compressed":
        return dict(ship_date=(p["ship"] - FRAME).to(torch.int16), quantity=p["qty"].to(torch.uint8),
                    extended_price=p["price"].to(torch.int32), discount=p["disc"], tax=p["tax"],
                    return_flag=_packed(p["rf"], 2), line_status=_packed(p["ls"], 1))
    wide = torch.int64 if layout == "reference" else torch.int8
    flags = torch.tensor(list(b"ANR"), dtype=torch.uint8, device="cuda")
    status = torch.tensor(list(b"FO"), dtype=torch.uint8, device="cuda")
    return dict(ship_date=p["ship"], quantity=(100 * p["qty"]).to(torch.int64 if layout == "reference" else torch.int32),
                extended_price=p["price"].to(torch.int64), discount=p["disc"].to(wide), tax=p["tax"].to(wide),
                return_flag=flags[p["rf"].long()], line_status=status[p["ls"].long()])


def _device_columns(layout, rows, seed, wide):
    parts = [_as_layout(layout, p) for _, p in _plain_rows(rows, seed, wide)]
    return {k: parts[0][k] if len(parts) == 1 else torch.cat([p[k] for p in parts]) for k in parts[0]}


def _pointers(cols):
    c = q1.Columns()
    for name, t in cols.items():
        setattr(c, name, t.data_ptr())
    return c


class _Owner:
    """Columns and the table that wraps them."""

    def __init__(self, layout, rows, seed, wide):
        self.cols = _device_columns(layout, rows, seed, wide)
        torch.cuda.synchronize()  # the library measures the columns on a stream of its own
        self.table = _context().wrap(LAYOUTS[layout], _pointers(self.cols), rows)


@functools.lru_cache(maxsize=None)
def _context():
    return q1.Context(0)


@functools.lru_cache(maxsize=None)
def _stream():
    return torch.cuda.Stream()


@functools.lru_cache(maxsize=None)
def _server():
    return serving.Server(_context())


def _requests(case, seed):
    """(table, seed of the table, rows of the table, first row, rows, cutoff) per request."""
    r = random.Random(seed)
    n, most = case["requests"], case["rows"]
    out = []
    if case["way"] == "batch":
        for i in range(n):
            rows = _log_uniform(r, min(10_000, most), most)
            out.append((i, seed * 1000 + i, rows, 0, rows, r.randint(CUTOFF_FIRST, CUTOFF_LAST)))
    else:
        sizes = np.geomspace(min(1_000_000, most / 2), most, 8).astype(int).tolist()
        for i in range(n):
            k = r.randrange(8)
            rows = r.randint(1, sizes[k])
            out.append((k, seed * 1000 + k, sizes[k], r.randint(0, sizes[k] - rows), rows,
                        r.randint(CUTOFF_FIRST, CUTOFF_LAST)))
    return out


# --- what a program holds, and one pass ------------------------------------------------------
class _Pinned:
    """Host columns in the library's pinned memory."""

    def __init__(self, layout, rows, seed):
        self.cols = _context().pinned_columns(LAYOUTS[layout], rows)
        for name, t in _device_columns(layout, rows, seed, False).items():
            kind = {2: np.int16, 4: np.int32}.get(t.element_size())
            to = self.cols[name].view(np.uint8 if kind is None else kind)
            torch.from_numpy(to).copy_(t.view(torch.uint8) if kind is None else t)

    def __del__(self):
        _context().free_pinned_columns(self.cols)


def prepare(case, seed):
    way, layout = case["way"], case["layout"]
    ctx = _context()
    cutoff = random.Random(seed).randint(CUTOFF_FIRST, CUTOFF_LAST)
    state = dict(case=case, ctx=ctx, cutoff=cutoff, placement=q1.PLACEMENTS[case["placement"]])
    if way in ("run", "pushdown"):
        state["owner"] = _Owner(layout, case["begin"] + case["rows"], seed, case["wide"])
    elif way in ("wrap", "enqueue"):
        state["cols"] = _device_columns(layout, case["rows"], seed, case["wide"])
        state["pointers"] = _pointers(state["cols"])
    elif way in ("batch", "serve"):
        reqs = _requests(case, seed)
        state["owners"] = owners = {}
        for k, s, rows, *_ in reqs:
            if k not in owners:
                owners[k] = _Owner(layout, rows, s, False)
        state["requests"] = [(owners[k].table, begin, rows, cut) for k, _, _, begin, rows, cut in reqs]
        if way == "batch":
            state["list"] = (q1.Request * len(reqs))(
                *[q1.Request(t.handle, begin, rows, cut, 0) for t, begin, rows, cut in state["requests"]])
            state["results"] = (q1.Result * len(reqs))()
        else:
            state["server"] = _server()
    else:
        state["pinned"] = _Pinned(layout, case["rows"], seed)
    torch.cuda.synchronize()
    return state


def _words(result):
    return np.frombuffer(result, dtype=np.int64).reshape(-1, q1.NUM_GROUPS, 8)


def _sums_as_words(groups):
    """(quantity, price, disc_price, charge, discount, count) per group as result words."""
    def pair(v):
        return [np.uint64(v & (1 << 64) - 1).astype(np.int64), v >> 64]

    return np.array([[q, p, *pair(dp), *pair(ch), d, n] for q, p, dp, ch, d, n in groups], dtype=np.int64)


def _group_words(groups):
    return _sums_as_words([(g.sum_qty, g.sum_base_price, g.sum_disc_price, g.sum_charge, g.sum_disc, g.count)
                           for g in groups])


def run(state):
    case, ctx, cutoff, placement = state["case"], state["ctx"], state["cutoff"], state["placement"]
    way, rows = case["way"], case["rows"]
    if way == "run":
        return _words(ctx.run_raw(state["owner"].table, case["begin"], rows, cutoff, placement))
    if way == "wrap":
        table = ctx.wrap(LAYOUTS[case["layout"]], state["pointers"], rows)
        result = ctx.run_raw(table, 0, rows, cutoff, placement)
        table.free()
        return _words(result)
    if way == "pushdown":
        table = ctx.build_filter(state["owner"].table, cutoff)
        result = ctx.run_raw(table, 0, rows, cutoff, placement)
        table.free()
        return _words(result)
    if way == "enqueue":
        with torch.cuda.stream(_stream()):
            sums = torch.zeros(8, q1.NUM_GROUPS, dtype=torch.int64, device="cuda")
            for first in range(0, rows, case["chunk"]):
                status = q1.lib.q1_enqueue(ctx.handle, placement, LAYOUTS[case["layout"]], None, sums.data_ptr(),
                                           ctypes.byref(state["pointers"]), first, min(case["chunk"], rows - first),
                                           cutoff, _stream().cuda_stream)
                ctx.check(status, "q1_enqueue")
        return sums
    if way == "batch":
        ctx.check(q1.lib.q1_run_batch(ctx.handle, state["list"], len(state["list"]), None, state["results"]),
                  "q1_run_batch")
        return _words(state["results"])
    if way == "serve":
        server, tickets, out = state["server"], [], []
        for table, begin, count, cut in state["requests"]:
            status, ticket = server.submit(table, begin, count, cut)
            ctx.check(status, "q1_server_submit")
            tickets.append(ticket)
        for ticket in tickets:
            status, groups, _ = server.wait(ticket)
            ctx.check(status, "q1_server_wait")
            out.append(_group_words(groups))
        return np.stack(out)
    return _group_words(ctx.run_streaming(LAYOUTS[case["layout"]], state["pinned"].cols, rows, cutoff, placement))


# --- what a pass cannot do without, and its exact result ---------------------------------------
def work(case):
    if case["way"] in ("batch", "serve"):
        rows = sum(r[4] for r in _requests(case, 1))
    else:
        rows = case["rows"]
    # per passing row: two subtractions or additions, two products and six sums
    return {"bytes": rows * BITS[case["layout"]] / 8, "flops": 10 * rows}


def _exact_words(rows, seed, wide, ranges):
    """The result words of each (first row, row after the last, cutoff) of one table."""
    total = [[[0] * 6 for _ in range(q1.NUM_GROUPS)] for _ in ranges]
    for r0, p in _plain_rows(rows, seed, wide):
        for i, (begin, end, cutoff) in enumerate(ranges):
            lo, hi = max(begin - r0, 0), min(end - r0, len(p["ship"]))
            for a in range(lo, hi, 1 << 24):
                c = {k: v[a:min(a + (1 << 24), hi)].long() for k, v in p.items()}
                slot = torch.where(c["ship"] <= cutoff, 2 * c["rf"] + c["ls"], -1)
                disc_price = (100 - c["disc"]) * c["price"]
                charge = disc_price * (100 + c["tax"])
                for g in range(q1.NUM_GROUPS):
                    m = slot == g
                    sums = [100 * c["qty"], c["price"], disc_price, charge, c["disc"], torch.ones_like(slot)]
                    got = torch.stack([s for v in sums for s in (((v >> 32) * m).sum(), ((v & 0xFFFFFFFF) * m).sum())])
                    got = got.tolist()
                    for f in range(6):
                        total[i][g][f] += (got[2 * f] << 32) + got[2 * f + 1]
    return [_sums_as_words(each) for each in total]


def exact(case, seed):
    way = case["way"]
    cutoff = random.Random(seed).randint(CUTOFF_FIRST, CUTOFF_LAST)
    if way in ("batch", "serve"):
        reqs = _requests(case, seed)
        out = [None] * len(reqs)
        for k in {r[0] for r in reqs}:
            mine = [i for i, r in enumerate(reqs) if r[0] == k]
            ranges = [(reqs[i][3], reqs[i][3] + reqs[i][4], reqs[i][5]) for i in mine]
            for i, words in zip(mine, _exact_words(reqs[mine[0]][2], reqs[mine[0]][1], False, ranges)):
                out[i] = words
        return np.stack(out)
    begin, end = case["begin"], case["begin"] + case["rows"]
    words = _exact_words(end, seed, case["wide"], [(begin, end, cutoff)])[0]
    if way == "enqueue":
        return torch.from_numpy(words.T.copy())
    return words[None] if way in ("run", "wrap", "pushdown") else words
