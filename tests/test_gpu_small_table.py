"""GPU parity of GROUP BY into tables whose keys fit a workgroup's LDS (the small-table kernel and
the one-pass kernel's copies), and of wide composite keys, against the oracle.  Integers are
bit-exact; floating SUM/AVG are FP64 sums of the same rows in another order: within 1e-12 relative
in FP64, and one rounding (1e-6) more where the output is FLOAT."""
import numpy as np
import pytest

import qikkdb_amd as qk
from gpu_util import Where, col, cpu_group_by, gpu_group_by
from helpers import as_map, maps_close

pytestmark = pytest.mark.gpu
ALL = [qk.AGG_SUM, qk.AGG_MIN, qk.AGG_MAX, qk.AGG_AVG, qk.AGG_COUNT, qk.AGG_COUNT_ALL]


def by_key(res, a):
    """as_map with NaN key parts named (NaN does not equal itself)."""
    return {tuple("nan" if x != x else x for x in k): v for k, v in as_map(res, a).items()}


def check(aggs, keys, vals, real, **kw):
    gkw = {k: kw.pop(k) for k in ("capacity", "flags", "path", "block", "tuning", "stats") if k in kw}
    got = gpu_group_by(aggs, keys, vals, **gkw, **kw)
    want = cpu_group_by(aggs, keys, vals, **kw)
    rel = (1e-6 if vals.dtype == np.float32 else 1e-12) if real else 0.0
    for a, agg in enumerate(aggs):
        maps_close(by_key(got, a), by_key(want, a), rel=rel if agg in (qk.AGG_SUM, qk.AGG_AVG) else 0.0)


# rows around a chunk of a wavefront (256), a workgroup's first round (2048) and several rounds
@pytest.mark.parametrize("n", [1, 255, 257, 2049, 70_001, 1_300_003])
@pytest.mark.parametrize("form", ["int", "long", "pair"])
@pytest.mark.parametrize("groups", [1, 15, 1000])
def test_small_table_forms(form, n, groups):
    rng = np.random.default_rng(n + groups)
    code = rng.integers(0, groups, n)
    vn, flags, kn, where, extra = rng.random(n) < 0.05, 0, None, (), None
    if form == "int":
        keys, vals = [(code * 7919 - 4000).astype(np.int32)], rng.lognormal(0, 1, n).astype(np.float32)
        kn = [rng.random(n) < 0.02]
        where = [Where(qk.GREATER_EQUAL, "value", 0.5, qk.FLOAT), Where(qk.LESS_EQUAL, "value", 4.0, qk.FLOAT)]
        aggs = [qk.AGG_SUM, qk.AGG_AVG, qk.AGG_COUNT]
    elif form == "long":
        keys = [(code.astype(np.int64) - groups // 2) * 0x123456789ABCD]
        keys[0][rng.random(n) < 0.03] = np.iinfo(np.int64).min  # the empty marker's bits
        kn, vals, aggs = [rng.random(n) < 0.02], rng.lognormal(0, 1, n), ALL
    else:
        keys = [(code % 7).astype(np.int32), (code // 7 - 2**31).astype(np.int32)]
        vals, aggs = rng.integers(-10**9, 10**9, n), [qk.AGG_SUM, qk.AGG_MIN, qk.AGG_MAX, qk.AGG_COUNT]
        extra = {"ts": (rng.integers(0, 1000, n).astype(np.int64), rng.random(n) < 0.1)}
        where, flags = [Where(qk.LESS, "ts", 600, qk.LONG)], qk.GB_KEYS_NOT_NULL
    check(aggs, keys, vals, vals.dtype.kind == "f", key_nulls=kn, value_nulls=vn, where=where, extra_cols=extra,
          capacity=groups + 2, flags=flags)


@pytest.mark.parametrize("copies_bytes", [-1, 8192])
def test_small_table_general_kernel(copies_bytes):
    """Forms the streaming reader does not take: a row mask, a FLOAT key, a predicate between columns."""
    rng = np.random.default_rng(3)
    n = 100_003
    vals = rng.integers(-1000, 1000, n)
    tuning = None if copies_bytes < 0 else {"lds_bytes": copies_bytes}
    fkey = (rng.integers(0, 40, n) * 0.5 - 10).astype(np.float32)
    check(ALL, [fkey], vals, False, mask=(rng.random(n) < 0.4).astype(np.int8), capacity=50, tuning=tuning)
    other = rng.integers(-1000, 1000, n)
    check(ALL, [rng.integers(0, 30, n).astype(np.int8)], vals, False, capacity=40, tuning=tuning,
          where=[Where(qk.GREATER, "value", rhs="other")], extra_cols={"other": (other, None)})


@pytest.mark.parametrize("cols", [2, 3, 4])
@pytest.mark.parametrize("groups,n", [(5, 300), (900, 50_001), (60_000, 1_200_007)])
def test_wide_composite_keys(cols, groups, n):
    """Nullable composite keys of two (INT, INT) to four key words (INT, LONG, DOUBLE, INT), in tables
    that fit the LDS and tables that do not; blocks of 2^18 rows, so later blocks find their keys."""
    rng = np.random.default_rng(cols * groups)
    code = rng.integers(0, groups, n)
    keys = [(code % 97 - 50).astype(np.int32), (code // 97).astype(np.int64 if cols > 2 else np.int32)]
    if cols > 2:
        keys.append(np.where(code % 5 == 0, np.nan, code % 11 * 0.5))
    if cols > 3:
        keys.append((code % 3).astype(np.int32))
    kn = [rng.random(n) < 0.03 for _ in keys]
    vals = rng.integers(-10**9, 10**9, n)
    check(ALL, keys, vals, False, key_nulls=kn, value_nulls=rng.random(n) < 0.05,
          capacity=max(64, 40 * groups), block=1 << 18)


@pytest.mark.parametrize("flags", [0, qk.GB_ASYNC])
@pytest.mark.parametrize("capacity", [64, 5000, 300_000, 3_000_000])
@pytest.mark.parametrize("form", ["plain", "mask", "value_range", "other_column", "mixed"])
def test_wide_keys_two_phase(form, capacity, flags):
    """Wide keys through the two phases over their slots, forced at every block size: one slot range up
    to several per partition, NULL keys and values, deferred and immediate merges, and every form of WHERE
    (rows it drops must not create groups)."""
    rng = np.random.default_rng(capacity + len(form))
    n, groups = 300_007, min(capacity // 2, 40_000)
    code = np.where(rng.random(n) < 0.5, rng.integers(0, 1 + groups // 50, n), rng.integers(0, groups, n))
    keys = [(code % 211 - 100).astype(np.int32), (code // 211).astype(np.int64)]
    kn = [rng.random(n) < 0.01, None] if capacity > 64 else None
    if kn is None:
        keys[0] = keys[0] * 0
    vals, vn = rng.lognormal(0, 1, n), rng.random(n) < 0.05
    other = rng.integers(0, 100, n).astype(np.int32)
    kw = {"extra_cols": {"other": (other, rng.random(n) < 0.05)}}
    if form == "mask":
        kw = {"mask": (rng.random(n) < 0.3).astype(np.int8)}
    elif form == "value_range":
        kw["where"] = [Where(qk.GREATER, "value", 0.5, qk.DOUBLE), Where(qk.LESS, "value", 4.0, qk.DOUBLE)]
    elif form == "other_column":
        kw["where"] = [Where(qk.LESS, "other", 40, qk.INT)]
    elif form == "mixed":
        kw["where"] = [Where(qk.NOT_EQUAL, "other", 7, qk.INT), Where(qk.GREATER, "value", 0.25, qk.DOUBLE)]
    stats = {}
    check(ALL, keys, vals, True, key_nulls=kn, value_nulls=vn, capacity=capacity, flags=flags, path=1,
          block=70_016, stats=stats, **kw)
    assert stats["path"] == 1 and stats["p1_form"] == 1


@pytest.mark.parametrize("flags", [0, qk.GB_ASYNC])
def test_wide_keys_without_scratch(flags):
    """A block of a wide-key table takes the one-pass kernel when the two phases' buffers cannot be had,
    also between blocks that have them."""
    rng = np.random.default_rng(5)
    n, block = 300_000, 100_000
    code = rng.integers(0, 30_000, n)
    keys, vals = [(code % 211).astype(np.int32), (code // 211).astype(np.int64)], rng.integers(-1000, 1000, n)
    kn = [rng.random(n) < 0.01, None]
    aggs = [qk.AGG_SUM, qk.AGG_MIN, qk.AGG_MAX, qk.AGG_COUNT]
    gb = qk.GPUGroupBy(aggs, [qk.INT, qk.LONG], qk.LONG, 40_000, 1, flags=flags)
    gb.set_path(1, 0)
    paths = []
    for at in range(0, n, block):
        part = slice(at, at + block)
        cols = [col(keys[0][part], kn[0][part]), col(keys[1][part]), col(vals[part])]
        try:
            if at == 0:
                qk._abi.call("qk_device_synchronize")
                qk._abi.call("qk_mem_release_cached")
                qk.set_memory_limit(qk.memory_stats()[0] + (1 << 20))
            gb.ProcessBlock([c.data for c in cols[:2]], cols[2].data, block, [c.nulls for c in cols[:2]], None)
        finally:
            qk.set_memory_limit(0)
        paths.append(gb.stats()["path"])
    got = gb.results_host()
    gb.close()
    want = cpu_group_by(aggs, keys, vals, key_nulls=kn)
    assert paths == [0, 1, 1]
    for a in range(len(aggs)):
        maps_close(by_key(got, a), by_key(want, a), rel=0.0)
