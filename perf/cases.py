"""The work a user of the WHERE -> reconstruct -> GROUP BY path has it do, at the sizes it is used at.

Sizes come from the reference engine's default block (262144 rows), from the benchmark's own
workloads (1M-row small query, 256M-row Zipf, 512M-row composite, the batched query mix) and from
the taxi queries the reference publishes (a handful of groups over very many rows).

A GROUP BY returns its groups in an unspecified order, so a program that shows them places each
at its key: every key here is a code in [0, groups) (a single int64 key carries it through an
odd multiplier, so that the keys are spread over 64 bits), and `run` scatters the result columns
into dense arrays by that code.
"""
import math

import numpy as np
import torch

import qikkdb_amd as qk
from qikkdb_amd.batch import BatchEngine, Query
from qikkdb_amd.strings import DeviceStrings, GPUGroupByString

DEV = "cuda"
TORCH_OF = {"int8": torch.int8, "int32": torch.int32, "int64": torch.int64, "float32": torch.float32,
            "float64": torch.float64}
QK_OF = {"int8": qk.INT8, "int32": qk.INT, "int64": qk.LONG, "float32": qk.FLOAT, "float64": qk.DOUBLE}
TYPESTR = {qk.INT8: "|i1", qk.INT: "<i4", qk.LONG: "<i8", qk.FLOAT: "<f4", qk.DOUBLE: "<f8"}
SIZE = {"int8": 1, "int32": 4, "int64": 8, "float32": 4, "float64": 8}
AGG = {"sum": qk.AGG_SUM, "avg": qk.AGG_AVG, "min": qk.AGG_MIN, "max": qk.AGG_MAX, "count": qk.AGG_COUNT}
OPS = {"gt": qk.GREATER, "ge": qk.GREATER_EQUAL, "lt": qk.LESS, "le": qk.LESS_EQUAL, "eq": qk.EQUAL, "ne": qk.NOT_EQUAL}
MIX = 0x9E3779B97F4A7C15          # odd: key = code * MIX mod 2^64, code = key * MIX^-1
UNMIX = pow(MIX, -1, 1 << 64)
TS0, DAY = 1735689600000, 86_400_000   # epoch milliseconds, one year of rows
YEAR = 365 * DAY
LO, HI = TS0 + 100 * DAY, TS0 + 130 * DAY  # the 30-day window of the WHERE on ts
CHUNK = 1 << 26


def _signed(x):
    return x - (1 << 64) if x >= 1 << 63 else x


# ---- the cases ----------------------------------------------------------------------------------

def listed():
    return [
        # one predicate over one block of the engine's default size: what the per-block loop of a
        # query does first; the call is latency
        {"name": "filter_block", "kind": "filter", "rows": 262_144, "type": "int32", "rhs": "const", "op": "gt",
         "nulls": 0.0},
        # the same over a whole resident column pair, one of them nullable
        {"name": "filter_columns", "kind": "filter", "rows": 100_000_007, "type": "float32", "rhs": "column",
         "op": "le", "nulls": 0.05},
        # the block's kept rows of one nullable column (reconstructColKeep)
        {"name": "compact_block", "kind": "compact", "rows": 262_139, "type": "int32", "keep": 0.5, "nulls": 0.1},
        # a whole column reconstructed by a mask that keeps a third of it
        {"name": "compact_column", "kind": "compact", "rows": 67_108_864, "type": "float64", "keep": 0.3,
         "nulls": 0.0},
        # SELECT a, v, ts WHERE ts in a month AND v > 0.5: filter and reconstruct fused
        {"name": "where_compact", "kind": "where", "rows": 30_000_001, "window": True, "nulls": 0.05},
        # the small query: 1M rows, 1000 groups, WHERE value > 0, SUM/MIN/MAX/COUNT
        {"name": "group_small", "kind": "group", "rows": 1 << 20, "blocks": 1, "key": "int32", "groups": 1000,
         "skew": 0.0, "value": "int32", "aggs": "sum,min,max,count", "where": "value", "nulls": 0.0, "fast": False},
        # SELECT passenger_count, AVG(total_amount), COUNT GROUP BY passenger_count: ten groups
        {"name": "group_taxi", "kind": "group", "rows": 200_000_000, "blocks": 3, "key": "int32", "groups": 10,
         "skew": 1.5, "value": "float32", "aggs": "avg,count", "where": "none", "nulls": 0.0, "fast": False},
        # 256M rows, Zipf keys over a million values, WHERE value BETWEEN, SUM/AVG/COUNT
        {"name": "group_zipf", "kind": "group", "rows": 1 << 28, "blocks": 4, "key": "int64", "groups": 1_000_000,
         "skew": 1.1, "value": "float32", "aggs": "sum,avg,count", "where": "value", "nulls": 0.05, "fast": True},
        # 512M rows, two int32 keys (16.7M groups), WHERE ts in a month, SUM/MIN/MAX/COUNT
        {"name": "group_composite", "kind": "group", "rows": 1 << 29, "blocks": 8, "key": "pair",
         "groups": 4096 * 4096, "skew": 0.0, "value": "int64", "aggs": "sum,min,max,count", "where": "ts",
         "nulls": 0.0, "fast": True},
        # two key columns, one of them nullable, and a nullable value: the engine's default columns
        {"name": "group_nullable", "kind": "group", "rows": 20_000_003, "blocks": 2, "key": "pair_null",
         "groups": 40_000, "skew": 0.8, "value": "int64", "aggs": "sum,min,max,count", "where": "none",
         "nulls": 0.05, "fast": False},
        # one string key column: a few hundred names, skewed
        {"name": "group_string", "kind": "string", "rows": 3_000_017, "groups": 700, "skew": 1.0, "nulls": 0.02},
        # many filtered GROUP BYs over one resident table in one run
        {"name": "batched", "kind": "batch", "rows": 1 << 27, "block": 1 << 22, "queries": 256, "mix": 7},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["filter", "compact", "where", "group", "group", "group", "group", "string", "batch"])
    nulls = rng.choice([0.0, 0.0, 0.02, 0.1])
    if kind == "filter":
        t = rng.choice(["int32", "int64", "float32", "float64"])
        # equality is asked of narrow integers; of reals and wide ones it holds for no row
        return {"kind": kind, "rows": _log(rng, 1 << 18, 1 << 27), "type": t, "rhs": rng.choice(["const", "column"]),
                "op": rng.choice(sorted(OPS) if t == "int32" else ["ge", "gt", "le", "lt"]), "nulls": nulls}
    if kind == "compact":
        return {"kind": kind, "rows": _log(rng, 1 << 18, 1 << 26), "type": rng.choice(["int8", "int32", "int64", "float32", "float64"]),
                "keep": round(rng.uniform(0.05, 0.95), 3), "nulls": nulls}
    if kind == "where":
        return {"kind": kind, "rows": _log(rng, 1 << 18, 1 << 26), "window": rng.random() < 0.5, "nulls": nulls}
    if kind == "string":
        return {"kind": kind, "rows": _log(rng, 1 << 16, 1 << 23), "groups": _log(rng, 20, 2000),
                "skew": rng.choice([0.0, 0.8, 1.1]), "nulls": nulls}
    if kind == "batch":
        return {"kind": kind, "rows": _log(rng, 1 << 24, 1 << 27), "block": 1 << rng.randint(18, 22),
                "queries": _log(rng, 32, 256), "mix": rng.randrange(1 << 20)}
    key = rng.choice(["int32", "int64", "int64", "pair", "pair_null"])
    rows = _log(rng, 1 << 16, 1 << 27)
    value = rng.choice(["int32", "int64", "float32", "float64"])
    return {"kind": "group", "rows": rows, "blocks": rng.choice([1, 1, 2, 4]), "key": key,
            "groups": _log(rng, 4, min(1 << 21, max(64, rows // 8))), "skew": rng.choice([0.0, 0.8, 1.1]),
            "value": value, "aggs": rng.choice(["sum,avg,count", "sum,min,max,count", "avg,count", "min,max,count"]),
            "where": rng.choice(["none", "value", "ts"]), "nulls": nulls, "fast": rng.random() < 0.5}


# ---- inputs -------------------------------------------------------------------------------------

def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 64 + stream)
    return g


def _codes(n, groups, skew, g):
    """int64 codes in [0, groups): uniform, or Zipf(skew) by inverse CDF with shuffled ranks."""
    if skew <= 0:
        return torch.randint(groups, (n,), generator=g, device=DEV)
    cdf = torch.arange(1, groups + 1, device=DEV, dtype=torch.float64).pow(-skew).cumsum(0)
    cdf /= cdf[-1].clone()
    order = torch.randperm(groups, generator=g, device=DEV)
    out = torch.empty(n, dtype=torch.int64, device=DEV)
    for at in range(0, n, CHUNK):
        u = torch.rand(min(CHUNK, n - at), generator=g, device=DEV, dtype=torch.float64)
        out[at:at + CHUNK] = order[torch.searchsorted(cdf, u).clamp_(max=groups - 1)]
    return out


def _values(n, kind, g):
    """lognormal(0, 1) reals, integers around zero."""
    t = TORCH_OF[kind]
    out = torch.empty(n, dtype=t, device=DEV)
    for at in range(0, n, CHUNK):
        part = out[at:at + CHUNK]
        if kind in ("float32", "float64"):
            part.normal_(generator=g).exp_()
        else:
            lim = 1_000_000_000 if kind == "int64" else 1000 if kind == "int32" else 100
            part.random_(-lim, lim + 1, generator=g)
    return out


def _times(n, g):
    out = torch.empty(n, dtype=torch.int64, device=DEV)
    return out.random_(TS0, TS0 + YEAR, generator=g)


def _isnull(n, p, g):
    if p <= 0:
        return None
    out = torch.empty(n, dtype=torch.bool, device=DEV)
    for at in range(0, n, CHUNK):
        out[at:at + CHUNK] = torch.rand(min(CHUNK, n - at), generator=g, device=DEV) < p
    return out


def _pack(isnull):
    """bool per row -> LSB-first bit mask of whole 64-bit words."""
    if isnull is None:
        return None
    n = isnull.numel()
    bits = torch.zeros((n + 63) // 64 * 64, dtype=torch.uint8, device=DEV)
    bits[:n] = isnull
    w = torch.tensor([1, 2, 4, 8, 16, 32, 64, 128], dtype=torch.uint8, device=DEV)
    return (bits.view(-1, 8) * w).sum(1, dtype=torch.uint8).view(torch.int64)


def _buf(t, byte_offset=0):
    return None if t is None else qk.DeviceBuffer(t.numel() * t.element_size() - byte_offset,
                                                  ptr=t.data_ptr() + byte_offset, owned=False)


def _col(t, kind, nulls=None, row=0, n=None):
    """Rows [row, row + n) of a tensor as a device column (row a multiple of 64)."""
    n = t.numel() - row if n is None else n
    return qk.DeviceColumn(_buf(t, row * t.element_size()), QK_OF[kind], n, _buf(nulls, row // 8))


class _View:
    """Device memory of the library, for torch; keeps its owner alive."""

    def __init__(self, buf, count, typestr):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": typestr, "data": (buf.ptr, False), "version": 2}


def _view(buf, count, qtype):
    return torch.as_tensor(_View(buf, count, TYPESTR[qtype]), device=DEV)


def _words(buf, rows):
    return _view(buf, (rows + 63) // 64, qk.LONG)


_SHIFTS = {}


def _bits(buf, rows):
    """A bit mask of the library as one bool per row."""
    if "s" not in _SHIFTS:
        _SHIFTS["s"] = torch.arange(64, device=DEV)
    return ((_words(buf, rows).view(-1, 1) >> _SHIFTS["s"]) & 1).view(-1)[:rows].bool()


# ---- filter -------------------------------------------------------------------------------------

def _filter_inputs(case, seed):
    n, kind = case["rows"], case["type"]
    a = _values(n, kind, _gen(seed, 1))
    b = _values(n, kind, _gen(seed, 2)) if case["rhs"] == "column" else None
    return a, b, _isnull(n, case["nulls"], _gen(seed, 3))


def _const(kind):
    return 1.25 if kind.startswith("float") else 10


def _prepare_filter(case, seed):
    a, b, isnull = _filter_inputs(case, seed)
    kind = case["type"]
    nulls = _pack(isnull)
    out = torch.empty(case["rows"], dtype=torch.int8, device=DEV)
    rhs = _col(b, kind) if b is not None else qk.Const(_const(kind), QK_OF[kind])
    return {"A": _col(a, kind), "B": rhs, "nulls": _buf(nulls), "out": _buf(out), "mask": out, "keep": (a, b, nulls)}


def _run_filter(case, s):
    qk.GPUBinary.Filter(OPS[case["op"]], s["A"], s["B"], case["rows"], s["nulls"], out=s["out"])
    return s["mask"]


def _exact_filter(case, seed):
    a, b, isnull = _filter_inputs(case, seed)
    m = getattr(torch, case["op"])(a, b if b is not None else _const(case["type"]))
    return (m if isnull is None else m & ~isnull).to(torch.int8)


# ---- reconstruct --------------------------------------------------------------------------------

def _exactly(mask, k):
    """The rows to change so that k of the mask's rows are set, spread over them: (set, to be cleared)
    or (clear, to be set)."""
    have = int(mask.sum())
    rows = (mask if have > k else ~mask).nonzero().view(-1)
    d = abs(have - k)
    return rows[torch.arange(d, device=DEV) * rows.numel() // max(d, 1)], have < k


def _compact_inputs(case, seed):
    n = case["rows"]
    col = _values(n, case["type"], _gen(seed, 1))
    mask = torch.rand(n, generator=_gen(seed, 2), device=DEV) < case["keep"]
    rows, up = _exactly(mask, round(n * case["keep"]))  # as many kept rows whatever the seed
    mask[rows] = up
    return col, mask, _isnull(n, case["nulls"], _gen(seed, 3))


def _prepare_compact(case, seed):
    col, keep, isnull = _compact_inputs(case, seed)
    mask, nulls = keep.to(torch.int8), _pack(isnull)
    return {"col": _buf(col), "mask": _buf(mask), "nulls": _buf(nulls), "keep": (col, mask, nulls)}


def _run_compact(case, s):
    kind = case["type"]
    out, count, nulls = qk.GPUReconstruct.reconstructColKeep(s["col"], SIZE[kind], s["mask"], case["rows"], s["nulls"])
    return {"values": _view(out, count, QK_OF[kind]), "nulls": None if nulls is None else _words(nulls, count)}


def _exact_compact(case, seed):
    col, keep, isnull = _compact_inputs(case, seed)
    out = col[keep]
    return {"values": out.double() if out.is_floating_point() else out,
            "nulls": None if isnull is None else _pack(isnull[keep])}


def _where_inputs(case, seed):
    n = case["rows"]
    a, v, ts = _values(n, "int32", _gen(seed, 1)), _values(n, "float64", _gen(seed, 2)), _times(n, _gen(seed, 3))
    isnull = _isnull(n, case["nulls"], _gen(seed, 4))
    rows, up = _exactly(_where_keeps(case, v, ts, isnull), round(n * _where_share(case)))
    v[rows] = 1.0 if up else 0.25  # as many passing rows whatever the seed
    if up:
        ts[rows] = LO
        if isnull is not None:
            isnull[rows] = False
    return a, v, ts, isnull


def _where_keeps(case, v, ts, isnull):
    keep = v > 0.5
    if case["window"]:
        keep &= (ts >= LO) & (ts < HI)
    return keep if isnull is None else keep & ~isnull


def _where_share(case):
    return 0.7559 * (1 - case["nulls"]) * (30 / 365 if case["window"] else 1)


def _prepare_where(case, seed):
    a, v, ts, isnull = _where_inputs(case, seed)
    nulls = _pack(isnull)
    cols = [_col(a, "int32"), _col(v, "float64", nulls), _col(ts, "int64")]
    preds = [qk.where(qk.GREATER, cols[1], qk.Const(0.5, qk.DOUBLE))]
    if case["window"]:
        preds += _window(cols[2])
    return {"cols": cols, "preds": preds, "keep": (a, v, ts, nulls)}


def _run_where(case, s):
    cols, count = qk.GPUReconstruct.WhereCompact(s["preds"], s["cols"], case["rows"])
    out = {"c%d" % i: _view(c.data, count, c.qtype) for i, c in enumerate(cols)}
    if cols[1].nulls is not None:
        out["nulls"] = _words(cols[1].nulls, count)
    return out


def _exact_where(case, seed):
    a, v, ts, isnull = _where_inputs(case, seed)
    keep = _where_keeps(case, v, ts, isnull)
    out = {"c0": a[keep], "c1": v[keep], "c2": ts[keep]}
    if isnull is not None:
        out["nulls"] = _pack(isnull[keep])
    return out


def _window(ts):
    return [qk.where(qk.GREATER_EQUAL, ts, qk.Const(LO, qk.LONG)), qk.where(qk.LESS, ts, qk.Const(HI, qk.LONG))]


# ---- GROUP BY -----------------------------------------------------------------------------------

def _sides(case):
    """(range of a, range of b) of a two-column key: code = a * range of b + b; a NULL `a` is the code
    after the last one of a."""
    b = max(1, math.isqrt(case["groups"]))
    return -(-case["groups"] // b), b


def _group_inputs(case, seed):
    n, key = case["rows"], case["key"]
    code = _codes(n, case["groups"], case["skew"], _gen(seed, 1))
    knull = None
    if key == "int32":
        keys = [code.to(torch.int32)]
    elif key == "int64":
        keys = [code * _signed(MIX)]
    else:
        ra, rb = _sides(case)
        a, b = (code // rb).to(torch.int32), (code % rb).to(torch.int32)
        keys = [a, b]
        if key == "pair_null":
            knull = _isnull(n, 0.03, _gen(seed, 4))
            code = torch.where(knull, ra * rb + b, code)
    value = _values(n, case["value"], _gen(seed, 2))
    ts = _times(n, _gen(seed, 5)) if case["where"] == "ts" else None
    return code, keys, knull, value, _isnull(n, case["nulls"], _gen(seed, 3)), ts


def _slots(case):
    if not case["key"].startswith("pair"):
        return case["groups"]
    ra, rb = _sides(case)
    return (ra + (case["key"] == "pair_null")) * rb


def _value_preds(col, kind):
    if kind.startswith("float"):
        return [qk.where(qk.GREATER_EQUAL, col, qk.Const(0.5, col.qtype)),
                qk.where(qk.LESS_EQUAL, col, qk.Const(4.0, col.qtype))]
    return [qk.where(qk.GREATER, col, qk.Const(0, col.qtype))]


def _prepare_group(case, seed):
    _, keys, knull, value, isnull, ts = _group_inputs(case, seed)
    kind, n = case["value"], case["rows"]
    nulls, knulls = _pack(isnull), _pack(knull)
    aggs = case["aggs"].split(",")
    kt = [qk.LONG if case["key"] == "int64" else qk.INT] * len(keys)
    flags = 0 if knull is not None else qk.GB_KEYS_NOT_NULL
    if case["fast"]:
        flags |= qk.GB_ASYNC
    slots = _slots(case)
    gb = qk.GPUGroupBy([AGG[a] for a in aggs], kt, QK_OF[kind], 1 << max(6, (slots - 1).bit_length()), 1, flags=flags)
    if case["fast"] and case["blocks"] > 4:
        gb.set_defer_rows(n)  # the whole query merges once
    step = -(-n // case["blocks"] // 64) * 64 if n % (64 * case["blocks"]) else n // case["blocks"]
    blocks = []
    for row in range(0, n, step):
        m = min(step, n - row)
        vcol = _col(value, kind, nulls, row, m)
        preds = []
        if case["where"] == "value":
            preds = _value_preds(vcol, kind)
        elif case["where"] == "ts":
            preds = _window(_col(ts, "int64", None, row, m))
        blocks.append((m, [_buf(k, row * k.element_size()) for k in keys],
                       None if knulls is None else [_buf(knulls, row // 8), None], vcol, preds))
    dense = [torch.zeros(slots, dtype=torch.int64 if a == "count" else TORCH_OF[kind], device=DEV) for a in aggs]
    return {"gb": gb, "blocks": blocks, "dense": dense, "flags": torch.zeros(slots, dtype=torch.bool, device=DEV),
            "aggs": aggs, "keep": (keys, knulls, value, nulls, ts)}


def _code_of(case, r, g):
    key = case["key"]
    if key == "int32":
        return _view(r.keys[0], g, qk.INT).long()
    if key == "int64":
        return _view(r.keys[0], g, qk.LONG) * _signed(UNMIX)
    ra, rb = _sides(case)
    a, b = _view(r.keys[0], g, qk.INT).long(), _view(r.keys[1], g, qk.INT)
    if key == "pair_null":
        a = torch.where(_bits(r.key_nulls[0], g), ra, a)
    return a * rb + b


def _run_group(case, s):
    gb = s["gb"]
    gb.reset()
    for m, keys, knulls, vcol, preds in s["blocks"]:
        if preds:
            gb.ProcessBlockWhere(keys, vcol.data, m, preds, knulls, vcol.nulls)
        else:
            gb.ProcessBlock(keys, vcol.data, m, knulls, vcol.nulls)
    # a NULL aggregate can only come from a nullable value column
    want = case["nulls"] > 0 or case["key"] == "pair_null"
    r = gb.GetResults(want_nulls=want)
    s["last"] = r  # its buffers stay until the next query's results replace them
    g = r.count
    code = _code_of(case, r, g)
    for dst, buf, t in zip(s["dense"], r.values, gb.out_types):
        dst.index_copy_(0, code, _view(buf, g, t))
    out = {"groups": g, "aggs": s["dense"]}
    if want:
        s["flags"].index_copy_(0, code, _bits(r.value_nulls[0], g))
        out["null"] = s["flags"]
    return out


def _by_code(code, value, slots, how="sum"):
    """Counts (value None), FP64 sums or extremes by code, 0 where no row has it: over several copies of
    the codes, one row in so many each, then over the copies (a frequent code's rows would queue)."""
    copies = max(1, min(65536, (1 << 25) // slots))
    init = {"sum": 0.0, "amin": float("inf"), "amax": float("-inf")}[how]
    out = torch.full((copies * slots,), init if value is not None else 0, device=DEV,
                     dtype=torch.int64 if value is None else torch.float64)
    for at in range(0, code.numel(), CHUNK):
        c = code[at:at + CHUNK]
        c = c + torch.arange(c.numel(), device=DEV) % copies * slots
        if value is None:
            out.index_add_(0, c, torch.ones_like(c))
        elif how == "sum":
            out.index_add_(0, c, value[at:at + CHUNK].double())
        else:
            out.scatter_reduce_(0, c, value[at:at + CHUNK].double(), how)
    out = out.view(copies, slots)
    out = out.sum(0) if how == "sum" else getattr(torch, how)(out, 0)
    return out if how == "sum" else torch.where(out.isinf(), 0.0, out)


def _exact_group(case, seed):
    code, _, _, value, isnull, ts = _group_inputs(case, seed)
    kind, slots = case["value"], _slots(case)
    real = kind.startswith("float")
    keep = None
    if case["where"] == "value":
        keep = (value >= 0.5) & (value <= 4.0) if real else value > 0
        if isnull is not None:
            keep &= ~isnull
    elif case["where"] == "ts":
        keep = (ts >= LO) & (ts < HI)
    if keep is not None:
        code, value = code[keep], value[keep]
        isnull = None if isnull is None else isnull[keep]
    rows = _by_code(code, None, slots)
    if isnull is not None:
        code, value = code[~isnull], value[~isnull]
    cnt = _by_code(code, None, slots)
    out = []
    for a in case["aggs"].split(","):
        if a == "count":
            out.append(cnt)
        elif a in ("sum", "avg") and real:
            sm = _by_code(code, value, slots)
            if a == "avg":
                sm = torch.where(cnt > 0, sm / cnt, torch.where(rows > 0, float("nan"), 0.0))
            out.append(sm)
        elif real and case["nulls"] == 0:
            out.append(_by_code(code, value, slots, "amin" if a == "min" else "amax"))
        else:
            out.append(None)  # whole numbers, or the limit of the type where every value is NULL
    return {"groups": int((rows > 0).sum()), "aggs": out}


# ---- GROUP BY a string ----------------------------------------------------------------------------

def _names(groups):
    """`groups` distinct names of 5 to 29 bytes."""
    r = np.random.default_rng(groups)
    letters = np.frombuffer(b"abcdefghijklmnopqrstuvwxyz -_", np.uint8)
    return [b"%04d%s" % (i, letters[r.integers(0, len(letters), r.integers(1, 26))].tobytes()) for i in range(groups)]


def _string_inputs(case, seed):
    n = case["rows"]
    code = _codes(n, case["groups"], case["skew"], _gen(seed, 1))
    code[:case["groups"]] = torch.arange(case["groups"], device=DEV)  # every name at least once
    return code, _values(n, "float64", _gen(seed, 2)), _isnull(n, case["nulls"], _gen(seed, 3))


def _prepare_string(case, seed):
    code, value, isnull = _string_inputs(case, seed)
    n, names = case["rows"], _names(case["groups"])
    lens = torch.tensor([len(x) for x in names], device=DEV)
    blob = torch.from_numpy(np.frombuffer(b"".join(names), np.uint8).copy()).to(DEV)
    first = lens.cumsum(0) - lens
    ends = lens[code].cumsum(0)
    total = int(ends[-1])
    chars = torch.empty(total, dtype=torch.uint8, device=DEV)
    step = 1 << 21
    for at in range(0, n, step):  # the bytes of every row's name, one after the other
        c = code[at:at + step]
        b0, b1 = (int(ends[at - 1]) if at else 0), int(ends[min(at + step, n) - 1])
        src = torch.repeat_interleave(first[c] - (ends[at:at + step] - lens[c]), lens[c])
        chars[b0:b1] = blob[src + torch.arange(b0, b1, device=DEV)]
    nulls = _pack(isnull)
    gb = GPUGroupByString([qk.AGG_SUM, qk.AGG_AVG, qk.AGG_COUNT], qk.DOUBLE, 1 << max(6, case["groups"].bit_length()), 1)
    return {"gb": gb, "col": DeviceStrings(_buf(chars), _buf(ends), n, total), "value": _buf(value),
            "nulls": _buf(nulls), "keep": (chars, ends, value, nulls)}


def _run_string(case, s):
    gb = s["gb"]
    gb.reset()
    gb.ProcessBlock(s["col"], s["value"], case["rows"], None, s["nulls"])
    r = gb.results_host()
    order = sorted(range(r["count"]), key=r["keys"].__getitem__)
    return {"names": np.frombuffer(b"\n".join(r["keys"][i] for i in order), np.uint8),
            "aggs": [v[order] for v in r["values"]], "null": r["value_nulls"][0][order]}


def _exact_string(case, seed):
    code, value, isnull = _string_inputs(case, seed)
    g = case["groups"]
    seen = _by_code(code, None, g) > 0
    if isnull is not None:
        code, value = code[~isnull], value[~isnull]
    cnt, sm = _by_code(code, None, g), _by_code(code, value, g)
    names = [x for x, y in zip(_names(g), seen.tolist()) if y]  # in sorted order: the number leads
    return {"names": np.frombuffer(b"\n".join(names), np.uint8), "aggs": [sm[seen], (sm / cnt)[seen], cnt[seen]],
            "null": (cnt == 0)[seen]}


# ---- many queries over one table ------------------------------------------------------------------

def _mix(case):
    """The benchmark's query mix: log-uniform block ranges, ts windows of 0.1 % to 50 %, log-uniform
    key ranges up to a million."""
    r = np.random.default_rng(case["mix"])
    nblocks = -(-case["rows"] // case["block"])
    out = []
    for _ in range(case["queries"]):
        length = int(min(nblocks, max(1, math.floor(math.exp(r.uniform(0, math.log(nblocks + 1)))))))
        first = int(r.integers(0, nblocks - length + 1))
        sel = float(r.uniform(0.001, 0.5))
        lo = TS0 + int(r.uniform(0, 1 - sel) * YEAR)
        out.append(Query(first, length, lo, lo + int(sel * YEAR), int(max(1, math.floor(10 ** r.uniform(0, 6))))))
    return out


def _prepare_batch(case, seed):
    n = case["rows"]
    a = torch.empty(n, dtype=torch.int32, device=DEV).random_(0, 4096, generator=_gen(seed, 1))
    b = torch.empty(n, dtype=torch.int32, device=DEV).random_(0, 4096, generator=_gen(seed, 2))
    ts, value = _times(n, _gen(seed, 3)), _values(n, "int64", _gen(seed, 4))
    torch.cuda.synchronize()  # the engine samples ts as it is made
    eng = BatchEngine(a.data_ptr(), b.data_ptr(), ts.data_ptr(), value.data_ptr(), n, case["block"], 4096)
    return {"eng": eng, "queries": _mix(case), "keep": (a, b, ts, value)}


def _run_batch(case, s):
    eng = s["eng"]
    eng.run(s["queries"])
    cnt, sm, mn, mx, offs = eng.results()
    total = int(offs[-1])
    out = {name: _view(qk.DeviceBuffer(total * 8, ptr=p, owned=False), total, qk.LONG)
           for name, p in (("count", cnt), ("sum", sm), ("min", mn), ("max", mx))}
    return out


# ---- the interface --------------------------------------------------------------------------------

_PREPARE = {"filter": _prepare_filter, "compact": _prepare_compact, "where": _prepare_where, "group": _prepare_group,
            "string": _prepare_string, "batch": _prepare_batch}
_RUN = {"filter": _run_filter, "compact": _run_compact, "where": _run_where, "group": _run_group,
        "string": _run_string, "batch": _run_batch}
_EXACT = {"filter": _exact_filter, "compact": _exact_compact, "where": _exact_where, "group": _exact_group,
          "string": _exact_string}


def prepare(case, seed):
    qk.ensure_device()
    s = _PREPARE[case["kind"]](case, seed)
    s["case"] = case
    return s


def run(state):
    return _RUN[state["case"]["kind"]](state["case"], state)


def exact(case, seed):
    f = _EXACT.get(case["kind"])  # a batch returns whole numbers only
    return None if f is None else f(case, seed)


def work(case):
    n, kind = case["rows"], case["kind"]
    nullb = n / 8 if case.get("nulls", 0) > 0 else 0
    if kind == "filter":
        e = SIZE[case["type"]] * (2 if case["rhs"] == "column" else 1)
        return {"bytes": n * (e + 1) + nullb, "flops": n}
    if kind == "compact":
        e = SIZE[case["type"]]
        # a kept row's element is read and written, the mask and bitmap read whole
        return {"bytes": n * (1 + 2 * e * case["keep"]) + nullb * (1 + case["keep"]), "flops": n}
    if kind == "where":
        # the predicates' columns are read whole, the other column and the outputs by the kept rows
        sel = _where_share(case)
        read = n * (16 + 4 * sel) if case["window"] else n * (8 + 12 * sel)
        return {"bytes": read + n * 20 * sel + nullb * (1 + sel), "flops": 2 * n}
    if kind == "string":
        return {"bytes": n * (8 + 8 + 17.0) + nullb, "flops": 20 * n}
    if kind == "batch":
        nblocks = -(-n // case["block"])
        pairs = groups = 0.0
        for q in _mix(case):
            last = min(q.first_block + q.nblocks, nblocks)
            pairs += min(last * case["block"], n) - q.first_block * case["block"]
            groups += q.key_mod
        return {"bytes": n * 24 + groups * 32, "flops": 2 * pairs}
    key = {"int32": 4, "int64": 8, "pair": 8, "pair_null": 8 + 1 / 8}[case["key"]]
    ts = 8 if case["where"] == "ts" else 0
    out = _slots(case) * (key + sum(8 if a == "count" else SIZE[case["value"]] for a in case["aggs"].split(",")))
    return {"bytes": n * (key + SIZE[case["value"]] + ts) + nullb + out, "flops": n * (1 + len(case["aggs"].split(",")))}
