"""The work a user of this engine has it do, as measurable cases.

Every case goes through the package's public entry points (buff_amd.Context,
Chunk, Batch, Server, SplitBDDoubleCompress) on columns of the kinds the
benchmark and the tests use: seeded random walks, uniform columns and
outlier-heavy columns, rounded to a number of decimals. Columns and outputs
are device tensors, except where a call takes host memory by its nature (the
codec on byte streams). All answers are whole numbers, bytes or float64 values
that the format fixes bit for bit, so every case is compared exactly.

Kinds:
  cycle   a column is encoded, queried once and dropped: encode, two range
          filters, equality, sum, max, decode at full and at reduced precision
          (what the reference's drivers time on one column);
  scan    the queries alone on a column that stays resident;
  batch   many uneven chunks resident; one call answers a mix of queries;
  ingest  many uneven chunks encoded in one call, their sums and maxima taken
          in a second one (zone maps), a few read back, then dropped;
  serve   a request trace, all arrivals at once, answered by the server;
  project filter one column, filter a second on the hits, gather its values;
  window  windowed maxima with their argmax rows;
  csv     text resident on the device to float64 values;
  codec   the reference-shaped calls on host arrays and host byte streams.
"""
import math

import numpy as np
import torch

import buff_amd
from buff_amd import _native as N

PRECISION_BITS = (0, 5, 8, 11, 15, 18, 21, 25, 28, 31, 35, 38, 50)   # fraction bits kept per decimals
LAYOUT = {"plain": 0, "slice": N.BUFF_SLICE, "major": N.BUFF_MAJORITY, "residue": N.BUFF_RESIDUE}

_context = None


def context():
    """One context for the process, as a program keeps one."""
    global _context
    if _context is None:
        _context = buff_amd.Context(0)
    return _context


# ---- the cases ------------------------------------------------------------------


def listed():
    return [
        # the smallest useful column (the batched workload's chunks start at 1024 rows): launches and waits count
        {"name": "cycle-walk-4k", "kind": "cycle", "data": "walk", "layout": "plain", "rows": 4097, "decimals": 4},
        # the 1M-row, 4-decimal walk that the reference's drivers are run on
        {"name": "cycle-walk-1m", "kind": "cycle", "data": "walk", "layout": "plain", "rows": 1 << 20, "decimals": 4},
        # an ordinary column whose rows tie with any predicate on the top byte almost everywhere; ragged length
        {"name": "cycle-uniform-17m", "kind": "cycle", "data": "uniform", "layout": "plain", "rows": 16777259,
         "decimals": 2},
        # outlier-heavy data in the sparse layout made for it
        {"name": "cycle-major-34m", "kind": "cycle", "data": "outlier", "layout": "major", "rows": 33554432,
         "decimals": 3},
        # the benchmark's largest column, resident, at 0.1 / 10 / 50 % selectivity
        {"name": "scan-walk-134m", "kind": "scan", "data": "walk", "rows": 134217728, "decimals": 4},
        # many small and middling chunks, a query mix over them in one call
        {"name": "batch-1024", "kind": "batch", "chunks": 1024, "low": 1024, "high": 1 << 20, "queries": 4096},
        # the same kind of chunks arriving: encoded together, statistics taken
        {"name": "ingest-512", "kind": "ingest", "chunks": 512, "low": 1024, "high": 1 << 20},
        # resident outlier-heavy chunks behind the server, saturated
        {"name": "serve-24", "kind": "serve", "chunks": 24, "low": 1 << 20, "high": 1 << 23, "requests": 512},
        # SELECT b WHERE a > p AND b > q
        {"name": "project-67m", "kind": "project", "rows": 67108864, "decimals": 4, "first": 0.5, "second": 0.2},
        # maxima of 1000-row windows (the data file's line length) over a whole column
        {"name": "window-34m", "kind": "window", "rows": 33554432, "decimals": 4, "window": 1000},
        # 1000 items a line, 4 decimals, as the reference's data file
        {"name": "csv-3m", "kind": "csv", "values": 3000000, "decimals": 4, "skip": 0},
        # a host program that keeps the reference's struct and its byte streams
        {"name": "codec-1m", "kind": "codec", "data": "uniform", "rows": 1 << 20, "decimals": 4},
    ]


def _log_between(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("cycle", "cycle", "cycle", "scan", "scan", "batch", "ingest", "serve", "project", "window",
                       "csv", "codec"))
    if kind == "cycle":
        layout = rng.choice(("plain", "plain", "slice", "major", "residue"))
        if layout in ("major", "residue"):
            return {"kind": kind, "data": "outlier" if layout == "major" else "spikes", "layout": layout,
                    "rows": _log_between(rng, 4096, 1 << 25), "decimals": rng.choice((2, 3, 4))}
        # the byte-slice readers take at most 32 bits a value
        return {"kind": kind, "data": rng.choice(("walk", "uniform")), "layout": layout,
                "rows": _log_between(rng, 1024, 1 << 26), "decimals": rng.randint(1, 4 if layout == "slice" else 5)}
    if kind == "scan":
        return {"kind": kind, "data": rng.choice(("walk", "uniform")), "rows": _log_between(rng, 1024, 1 << 27),
                "decimals": rng.randint(1, 5)}
    if kind == "batch":
        return {"kind": kind, "chunks": _log_between(rng, 16, 1024), "low": 1024,
                "high": _log_between(rng, 1 << 14, 1 << 20), "queries": _log_between(rng, 32, 4096)}
    if kind == "ingest":
        return {"kind": kind, "chunks": _log_between(rng, 16, 512), "low": 1024,
                "high": _log_between(rng, 1 << 14, 1 << 20)}
    if kind == "serve":
        low = _log_between(rng, 1 << 14, 1 << 20)
        return {"kind": kind, "chunks": rng.randint(4, 24), "low": low, "high": 8 * low,
                "requests": _log_between(rng, 32, 512)}
    if kind == "project":
        return {"kind": kind, "rows": _log_between(rng, 4096, 1 << 26), "decimals": rng.randint(1, 5),
                "first": rng.uniform(0.05, 0.9), "second": rng.uniform(0.001, 0.5)}
    if kind == "window":
        rows = _log_between(rng, 4096, 1 << 25)
        return {"kind": kind, "rows": rows, "decimals": rng.randint(1, 5), "window": _log_between(rng, 7, rows)}
    if kind == "csv":
        return {"kind": kind, "values": _log_between(rng, 1000, 3000000), "decimals": rng.randint(1, 6),
                "skip": rng.choice((0, 1))}
    return {"kind": "codec", "data": "uniform", "rows": _log_between(rng, 1000, 1 << 20),
            "decimals": rng.randint(1, 5)}


# ---- columns --------------------------------------------------------------------


def _generator(seed, salt=0):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1009 + salt)


def _decimals(k, unit):
    """k / unit, correctly rounded (a division by a Python number would multiply by its reciprocal)."""
    return k.to(torch.float64).div_(torch.tensor(float(unit), dtype=torch.float64, device="cuda"))


def column(data, rows, decimals, seed, salt=0):
    """A float64 device column of values with `decimals` decimals. The decimal units are whole numbers (sums of whole
    numbers are the same in any order), divided once."""
    g = _generator(seed, salt)
    unit = 10 ** decimals

    def normal():
        return torch.randn(rows, generator=g, device="cuda", dtype=torch.float64)

    def rand():
        return torch.rand(rows, generator=g, device="cuda", dtype=torch.float64)

    if data == "walk":        # x0 = 0, N(0, 1) steps
        k = (normal() * unit).round_().to(torch.int64)
        k[0] = 0
        k = k.cumsum(0)
    elif data == "uniform":   # U[-1000, 1000]
        k = ((rand() * 2000.0 - 1000.0) * unit).round_().to(torch.int64)
    elif data == "outlier":   # 95% N(100, 0.5), 5% +-10^U[6, 9]
        x = 100.0 + 0.5 * normal()
        hit = rand() < 0.05
        far = 10.0 ** (6.0 + 3.0 * rand())
        x = torch.where(hit, torch.where(rand() < 0.5, -far, far), x)
        k = (x * unit).round_().to(torch.int64)
    else:                     # "spikes": 99% N(100, 0.5), 1% 100 + 10^U[3, 7]
        x = 100.0 + 0.5 * normal()
        x = torch.where(rand() < 0.01, 100.0 + 10.0 ** (3.0 + 4.0 * rand()), x)
        k = (x * unit).round_().to(torch.int64)
    return _decimals(k, unit)


def values_above(x, shares):
    """For each share, a value of the column with about that share of the rows above it."""
    step = max(1, x.numel() // 1000003)
    s = x[::step].sort().values
    return [float(s[min(s.numel() - 1, int((1.0 - q) * s.numel()))]) for q in shares]


def stored(x, decimals):
    """The fixed-point values the format keeps of a column: truncated to the fraction bits of its decimals."""
    scale = 2.0 ** PRECISION_BITS[decimals]
    return (x * scale).trunc() / scale


def _words(rows):
    return torch.zeros((rows + 63) // 64, dtype=torch.int64, device="cuda")


def _uneven(case):
    """Row offsets and decimals of uneven chunks, lengths log-uniform: the case's own, so that outputs have the same
    shapes for every seed (the values are the seed's)."""
    r = np.random.default_rng([case["chunks"], case["low"], case["high"]])
    lens = np.exp(r.uniform(np.log(case["low"]), np.log(case["high"]), case["chunks"])).astype(np.int64)
    off = np.concatenate([[0], np.cumsum(lens)])
    return off, r.integers(1, 7, case["chunks"]), r


class _Memory:
    """Device memory that the engine owns, for torch.as_tensor."""

    def __init__(self, ptr, count, kind):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": (count,), "typestr": kind, "version": 2}


def _results(res):
    return np.frombuffer(res._res, dtype=N.RESULT_DTYPE)[: len(res)]


# ---- prepare / run --------------------------------------------------------------


def prepare(case, seed):
    state = {"case": case}
    PREPARE[case["kind"]](state, case, seed)
    torch.cuda.synchronize()   # the engine works on streams of its own
    return state


def run(state):
    return RUN[state["case"]["kind"]](state, state["case"])


def _prepare_cycle(s, case, seed):
    rows = case["rows"]
    s["x"] = column(case["data"], rows, case["decimals"], seed)
    s["preds"] = values_above(s["x"], (0.1, 0.5)) + [float(s["x"][rows // 3])]
    s["bitmaps"] = [_words(rows) for _ in s["preds"]]
    s["full"] = torch.zeros(rows, dtype=torch.float64, device="cuda")
    s["part"] = torch.zeros(rows, dtype=torch.float64, device="cuda")
    context()


def _run_cycle(s, case):
    layout = case["layout"]
    semantic = N.BUFF_SEMANTIC if layout == "residue" else 0
    ch = context().encode_device(s["x"].data_ptr(), case["rows"], 10 ** case["decimals"], flags=LAYOUT[layout])
    for op, pred, words in zip(("range", "range", "equal"), s["preds"], s["bitmaps"]):
        ch.filter_device(op, pred, words.data_ptr(), flags=semantic)
    ref, exact, sums = ch.sum()
    top = ch.max_ex(flags=semantic)
    info = ch.info()
    ch.materialize_device(s["full"].data_ptr())
    out = {"bitmaps": s["bitmaps"], "reference_sum": ref, "sum": exact, "column_sums": sums, "max": top[0],
           "max_offset": top[1], "header": [info.base, info.n, info.ilen, info.dlen], "full": s["full"]}
    if layout != "slice":   # the byte-slice format has no reduced-precision decode
        ch.materialize_device(s["part"].data_ptr(), max(case["decimals"] - 2, 0), flags=N.BUFF_SEMANTIC)
        out["part"] = s["part"]
    ch.free()
    return out


def _prepare_scan(s, case, seed):
    rows = case["rows"]
    x = column(case["data"], rows, case["decimals"], seed)
    s["preds"] = values_above(x, (0.001, 0.1, 0.5)) + [float(x[rows // 3])]
    s["bitmaps"] = [_words(rows) for _ in s["preds"]]
    torch.cuda.synchronize()
    s["chunk"] = context().encode_device(x.data_ptr(), rows, 10 ** case["decimals"])
    context().synchronize()


def _run_scan(s, case):
    ch = s["chunk"]
    for op, pred, words in zip(("range", "range", "range", "equal"), s["preds"], s["bitmaps"]):
        ch.filter_device(op, pred, words.data_ptr())
    ref, exact, sums = ch.sum()
    top = ch.max()
    return {"bitmaps": s["bitmaps"], "reference_sum": ref, "sum": exact, "column_sums": sums, "max": top[0],
            "max_offset": top[1]}


def _uneven_column(case, seed):
    """Walks of several decimals end to end: (x, row offsets, scales, the generator)."""
    off, decimals, r = _uneven(case)
    x = column("walk", int(off[-1]), 6, seed)
    unit = torch.repeat_interleave(torch.from_numpy(10.0 ** decimals.astype(np.float64)),
                                   torch.from_numpy(np.diff(off))).cuda()
    x = (x * unit).round_().div_(unit)
    return x, off.astype(np.uint64), (10 ** decimals).astype(np.uint64), r


def _prepare_batch(s, case, seed):
    x, off, scales, r = _uneven_column(case, seed)
    torch.cuda.synchronize()
    s["batch"] = context().batch_encode_device(x.data_ptr(), off, scales)
    nq = case["queries"]
    lens = np.diff(off.astype(np.int64))
    chunk = r.integers(0, case["chunks"], nq)
    row = off[chunk].astype(np.int64) + (r.random(nq) * lens[chunk]).astype(np.int64)
    pred = x[torch.from_numpy(row).cuda()].cpu().numpy()
    op = np.array([N.BUFF_Q_EQ, N.BUFF_Q_GT, N.BUFF_Q_SUM, N.BUFF_Q_MAX])[r.integers(0, 4, nq)]
    op[r.random(nq) < 1.0 / 64] = N.BUFF_Q_MAT
    s["queries"] = N.prepare_queries([(int(o), int(c), float(p), -1, 0) for o, c, p in zip(op, chunk, pred)])
    # where the outputs lie in the batch's arena: the words of every bitmap and value, without the padding between
    res = _results(s["batch"].query(s["queries"]))
    at, count = [], []
    for o, c, where in zip(op, chunk, res["out_offset"]):
        if o in (N.BUFF_Q_EQ, N.BUFF_Q_GT):
            at.append(int(where) // 8)
            count.append((int(lens[c]) + 63) // 64)
        elif o == N.BUFF_Q_MAT:
            at.append(int(where) // 8)
            count.append(int(lens[c]))
    count = torch.tensor(count or [0], device="cuda")
    at = torch.tensor(at or [0], device="cuda")
    begin = count.cumsum(0) - count
    s["index"] = torch.arange(int(count.sum()), device="cuda") + torch.repeat_interleave(at - begin, count)
    s["words"] = int(s["index"].max()) + 1 if s["index"].numel() else 0


def _run_batch(s, case):
    res = _results(s["batch"].query(s["queries"]))
    out = {"status": res["status"], "count": res["count"].view(np.int64), "value": res["value"],
           "exact": res["exact"], "max_offset": res["max_off"].view(np.int64)}
    if s["words"]:
        arena = torch.as_tensor(_Memory(s["batch"].arena()[0], s["words"], "<i8"), device="cuda")
        out["outputs"] = arena[s["index"]]
    return out


def _prepare_ingest(s, case, seed):
    s["x"], s["off"], s["scales"], _ = _uneven_column(case, seed)
    s["queries"] = N.prepare_queries([(op, c, 0.0, -1, 0) for c in range(case["chunks"])
                                      for op in (N.BUFF_Q_SUM, N.BUFF_Q_MAX)])
    # four of the chunks are read back
    lens = np.diff(s["off"].astype(np.int64))
    s["back"] = [(int(c), torch.zeros(int(lens[c]), dtype=torch.float64, device="cuda"))
                 for c in np.linspace(0, case["chunks"] - 1, 4).astype(int)]
    context()


def _run_ingest(s, case):
    batch = context().batch_encode_device(s["x"].data_ptr(), s["off"], s["scales"])
    res = _results(batch.query(s["queries"]))
    for c, values in s["back"]:
        batch.chunks[c].materialize_device(values.data_ptr())
    batch.free()
    return {"status": res["status"], "value": res["value"], "exact": res["exact"],
            "max_offset": res["max_off"].view(np.int64), "values": [values for _, values in s["back"]]}


class _Served:
    """A server and the chunks it answers from, ended in that order."""

    def __init__(self, chunks):
        self.chunks = chunks
        self.server = buff_amd.Server(context(), max_batch=4096, slots=2, arena_bytes=1 << 20)
        for ch in chunks:
            self.server.add_chunk(ch)

    def __del__(self):
        self.server.destroy()
        for ch in self.chunks:
            ch.free()


def _prepare_serve(s, case, seed):
    off, _, r = _uneven(case)
    lens = np.diff(off)
    chunks = []
    for i, rows in enumerate(lens):
        x = column("outlier", int(rows), 3, seed, 1 + i)
        torch.cuda.synchronize()
        chunks.append(context().encode_device(x.data_ptr(), int(rows), 1000, flags=N.BUFF_MAJORITY))
        context().synchronize()
    s["served"] = _Served(chunks)
    # the request mix of the served workload: 60% range filters, 25% sums, 15% decodes at 1-3 decimals
    queries, words, values = [], [], []
    for u, k, p, d in zip(r.random(case["requests"]), r.integers(0, len(chunks), case["requests"]),
                          r.choice((99.5, 100.0, 100.5, 1e6), case["requests"]),
                          r.integers(1, 4, case["requests"])):
        n = int(lens[k])
        queries.append((N.BUFF_Q_GT, int(k), float(p), -1, 0) if u < 0.6 else
                       (N.BUFF_Q_SUM, int(k), 0.0, -1, 0) if u < 0.85 else
                       (N.BUFF_Q_MAT, int(k), 0.0, int(d), N.BUFF_SEMANTIC))
        words.append((n + 63) // 64 if u < 0.6 else 0)
        values.append(n if u >= 0.85 else 0)
    s["queries"] = N.prepare_queries(queries)
    s["arrival"] = np.zeros(case["requests"])
    s["bitmaps"] = torch.zeros(max(1, sum(words)), dtype=torch.int64, device="cuda")
    s["values"] = torch.zeros(max(1, sum(values)), dtype=torch.float64, device="cuda")
    wat, vat, outs = 0, 0, []
    for w, v in zip(words, values):
        outs.append(s["bitmaps"].data_ptr() + 8 * wat if w else s["values"].data_ptr() + 8 * vat if v else None)
        wat, vat = wat + w, vat + v
    s["outs"] = outs


def _run_serve(s, case):
    res, _ = s["served"].server.run_trace(s["queries"], s["arrival"], outs=s["outs"])
    res = _results(res)
    return {"status": res["status"], "count": res["count"].view(np.int64), "value": res["value"],
            "exact": res["exact"], "bitmaps": s["bitmaps"], "values": s["values"]}


def _prepare_project(s, case, seed):
    rows = case["rows"]
    a = column("walk", rows, case["decimals"], seed, 1)
    b = column("uniform", rows, 2, seed, 2)
    s["preds"] = values_above(a, (case["first"],)) + values_above(b, (case["second"],))
    torch.cuda.synchronize()
    s["a"] = context().encode_device(a.data_ptr(), rows, 10 ** case["decimals"])
    s["b"] = context().encode_device(b.data_ptr(), rows, 100)
    context().synchronize()
    s["first"], s["second"] = _words(rows), _words(rows)
    s["values"] = torch.zeros(rows, dtype=torch.float64, device="cuda")


def _run_project(s, case):
    a, b = s["a"], s["b"]
    a.filter_device("range", s["preds"][0], s["first"].data_ptr())
    b.filter_cond_device("range", s["preds"][1], s["first"].data_ptr(), s["second"].data_ptr())
    rows = b.materialize_cond_device(s["second"].data_ptr(), s["values"].data_ptr(), case["rows"],
                                     flags=N.BUFF_SEMANTIC)
    return {"first": s["first"], "second": s["second"], "rows": rows, "values": s["values"]}   # zeros after `rows`


def _prepare_window(s, case, seed):
    rows = case["rows"]
    x = column("walk", rows, case["decimals"], seed)
    torch.cuda.synchronize()
    s["chunk"] = context().encode_device(x.data_ptr(), rows, 10 ** case["decimals"])
    context().synchronize()
    s["argmax"] = _words(rows)
    s["values"] = torch.zeros(-(-rows // case["window"]), dtype=torch.float64, device="cuda")


def _run_window(s, case):
    k = s["chunk"].max_range_device(0, case["rows"], case["window"], s["values"].data_ptr(), s["values"].numel(),
                                    argmax_dev=s["argmax"].data_ptr(), flags=N.BUFF_SEMANTIC)
    return {"values": s["values"][:k], "argmax": s["argmax"]}


CSV_LINE = 1000


def _csv_units(case, seed):
    g = _generator(seed)
    k = (torch.randn(case["values"], generator=g, device="cuda", dtype=torch.float64) * 10 ** case["decimals"])
    k = k.round_().to(torch.int64)
    k[0] = 0
    return k.cumsum(0)


def _prepare_csv(s, case, seed):
    n, d = case["values"], case["decimals"]
    k = _csv_units(case, seed)
    mag = k.abs()
    digits = max(int(mag.max()), 1)
    width = max(len(str(digits)), d + 1)   # digits, at least one before the point
    # columns: sign, `width` digits with the point before the last d, separator
    text = torch.zeros((n, width + 3), dtype=torch.uint8, device="cuda")
    keep = torch.ones((n, width + 3), dtype=torch.bool, device="cuda")
    text[:, 0] = ord("-")
    keep[:, 0] = k < 0
    for j in range(width):
        power = 10 ** (width - 1 - j)
        at = 1 + j + (1 if j >= width - d else 0)
        text[:, at] = ((mag // power) % 10 + ord("0")).to(torch.uint8)
        if j < width - d - 1:   # no leading zeros
            keep[:, at] = mag >= power
    text[:, 1 + width - d] = ord(".")
    text[:, -1] = ord(",")
    text[CSV_LINE - 1::CSV_LINE, -1] = ord("\n")
    s["text"] = text[keep]
    s["values"] = torch.zeros(n, dtype=torch.float64, device="cuda")
    context()


def _run_csv(s, case):
    count = context().csv_parse_device(s["text"].data_ptr(), s["text"].numel(), s["values"].data_ptr(),
                                       s["values"].numel(), skip_val=case["skip"])
    return {"values": s["values"][:count]}


def _prepare_codec(s, case, seed):
    s["x"] = column(case["data"], case["rows"], case["decimals"], seed).cpu().numpy()
    s["pred"] = float(np.quantile(s["x"], 0.9, method="lower"))
    s["codec"] = buff_amd.SplitBDDoubleCompress(case["rows"], 1, 10 ** case["decimals"])


def _run_codec(s, case):
    codec = s["codec"]
    stream = codec.byte_fixed_encode(s["x"])
    words, count = codec.buff_range_filter(stream, s["pred"])
    return {"stream": stream, "words": words.view(np.int32), "count": count, "sum": codec.byte_fixed_sum(stream),
            "max": codec.byte_fixed_max(stream), "values": codec.byte_fixed_decode(stream)}


PREPARE = {"cycle": _prepare_cycle, "scan": _prepare_scan, "batch": _prepare_batch, "ingest": _prepare_ingest,
           "serve": _prepare_serve, "project": _prepare_project, "window": _prepare_window, "csv": _prepare_csv,
           "codec": _prepare_codec}
RUN = {"cycle": _run_cycle, "scan": _run_scan, "batch": _run_batch, "ingest": _run_ingest, "serve": _run_serve,
       "project": _run_project, "window": _run_window, "csv": _run_csv, "codec": _run_codec}


# ---- work, tolerance, exact -----------------------------------------------------


def _width(data, rows, decimals):
    """About the stored bits of a value."""
    span = {"walk": 2.0 * math.sqrt(max(rows, 2)), "uniform": 2000.0, "outlier": 2e9, "spikes": 1e7}[data]
    return math.ceil(math.log2(span)) + PRECISION_BITS[decimals]


def work(case):
    """Bytes that a pass cannot do without: each operation's input read once and its output written once."""
    kind, rows = case["kind"], case.get("rows", 0)
    if kind in ("cycle", "scan"):
        f = _width(case["data"], rows, case["decimals"]) / 8.0
        # an outlier-heavy column's sparse layout keeps 5% of its top bytes
        f -= {"major": 3 - 3 * 0.175, "residue": 2 - 2 * 0.135}.get(case.get("layout"), 0)
        query = 1.125
        if kind == "scan":
            return {"bytes": rows * (4 * query + f + 1), "flops": 0}
        # encode, three filters, sum, max, decode, decode at two decimals fewer
        part = 0 if case["layout"] == "slice" else 8 + f - 0.75
        return {"bytes": rows * (8 + f + 3 * query + f + 1 + f + 8 + part), "flops": 0}
    if kind in ("batch", "ingest", "serve"):
        mean = (case["high"] - case["low"]) / math.log(case["high"] / case["low"])
        f = 3.3 if kind != "serve" else (42 / 8.0 - 3 + 3 * 0.175)
        if kind == "ingest":   # encode, then a sum and a max of each chunk
            return {"bytes": case["chunks"] * mean * (8 + f + f + 1), "flops": 0}
        if kind == "batch":    # half filters, a quarter sums, a quarter maxima, one in 64 a decode
            return {"bytes": case["queries"] * mean * (0.5 * 1.125 + 0.25 * f + 0.25 + (8 + f) / 64), "flops": 0}
        return {"bytes": case["requests"] * mean * (0.6 * 1.6 + 0.25 * f + 0.15 * (8 + f)), "flops": 0}
    if kind == "project":
        hits = case["first"] * case["second"]
        return {"bytes": rows * (1.125 + 0.25 + case["first"] + 0.125 + hits * (19 / 8.0 + 8)), "flops": 0}
    if kind == "window":
        return {"bytes": rows * (_width("walk", rows, case["decimals"]) / 8.0 + 0.125) + 8.0 * rows / case["window"],
                "flops": 0}
    if kind == "csv":
        return {"bytes": case["values"] * (case["decimals"] + 6 + 8.0), "flops": 0}
    f = _width(case["data"], rows, case["decimals"]) / 8.0
    return {"bytes": rows * (8 + f + 4 * f + 0.125 + 8), "flops": 0}


def tolerance(case):
    """Bitmaps, counts, streams and offsets are whole numbers; decoded values, sums and maxima are fixed bit for bit
    by the format (exact integers rounded once, or the reference's fold replayed in its order)."""
    return "exact"


def exact(case, seed):
    """The values that 64-bit arithmetic gives where an output is one; None for bitmaps, counts and the reference's
    own quirks."""
    kind = case["kind"]
    if kind in ("cycle", "scan", "codec"):
        v = stored(column(case["data"], case["rows"], case["decimals"], seed), case["decimals"])
        out = {"sum": float(v.sum()), "max": float(v.max())}
        if kind == "cycle":
            out["full"] = v
            if case["layout"] == "major":   # the reference's decode and max of sparse columns are not the values
                out["full"] = out["max"] = None
        if kind == "codec":
            out["sum"], out["values"] = None, v.cpu().numpy()
        return out
    if kind == "project":
        a = column("walk", case["rows"], case["decimals"], seed, 1)
        b = column("uniform", case["rows"], 2, seed, 2)
        p = values_above(a, (case["first"],)) + values_above(b, (case["second"],))
        b = stored(b, 2)
        p = stored(torch.tensor([p[0]], dtype=torch.float64), case["decimals"]), \
            stored(torch.tensor([p[1]], dtype=torch.float64), 2)
        v = b[(stored(a, case["decimals"]) > float(p[0])) & (b > float(p[1]))]
        return {"values": torch.cat([v, torch.zeros(case["rows"] - len(v), dtype=torch.float64, device="cuda")])}
    if kind == "window":
        v = stored(column("walk", case["rows"], case["decimals"], seed), case["decimals"])
        w = case["window"]
        short = -len(v) % w
        v = torch.cat([v, torch.full((short,), -math.inf, dtype=torch.float64, device="cuda")])
        return {"values": v.reshape(-1, w).max(1).values}
    if kind == "csv":
        v = _decimals(_csv_units(case, seed), 10 ** case["decimals"])
        if case["skip"]:
            v = torch.cat([line[case["skip"]:] for line in v.split(CSV_LINE)])
        return {"values": v}
    return None
