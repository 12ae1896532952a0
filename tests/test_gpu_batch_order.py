"""The batch engine's ts-ordered copy against numpy, bit-exact: tables whose rows, blocks and tiles are no
multiples of a chunk, key numbers beyond 32 bits, ts in order and with few distinct values, windows that
end on values present, windows at the ends of the type, and empty ones."""
import numpy as np
import pytest

import qikkdb_amd as qk
from qikkdb_amd import batch as B

pytestmark = pytest.mark.gpu
I64 = np.iinfo(np.int64)


def expect(d, q, block, rows, b_range):
    r0, r1 = q.first_block * block, min((q.first_block + q.nblocks) * block, rows)
    a, b, ts, v = (d[k][r0:r1] for k in ("a", "b", "ts", "value"))
    m = (ts >= q.ts_lo) & (ts < q.ts_hi)
    key = (a[m].astype(np.int64) * b_range + b[m]) % q.key_mod
    cnt, sm = np.bincount(key, minlength=q.key_mod), np.zeros(q.key_mod, np.int64)
    mn, mx = np.full(q.key_mod, I64.max), np.full(q.key_mod, I64.min)
    np.add.at(sm, key, v[m])
    np.minimum.at(mn, key, v[m])
    np.maximum.at(mx, key, v[m])
    return cnt, sm, mn, mx


@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("rows,block,tile", [(100_003, 30_000, 8192), (65_536, 4096, 4096), (300_001, 300_001, 1 << 16)])
@pytest.mark.parametrize("form", ["plain", "wide", "time_ordered", "few_ts"])
def test_ordered_batch(form, rows, block, tile, graph):
    rng = np.random.default_rng(rows + len(form))
    lim = 2**31 - 1 if form == "wide" else 4096
    a = rng.integers(-lim if form == "wide" else 0, lim, rows).astype(np.int32)
    b = rng.integers(-50 if form == "wide" else 0, 4096, rows).astype(np.int32)
    if form == "wide":
        a[: rows // 2] = np.abs(a[: rows // 2]) % 4096  # tiles of both kinds
        b[: rows // 2] = np.abs(b[: rows // 2])
    ts = rng.integers(0, 10**6, rows)
    if form == "time_ordered":
        ts = np.sort(ts)
    if form == "few_ts":
        ts = rng.choice(np.array([I64.min, -5, 0, 7, I64.max]), rows)
    d = {"a": a, "b": b, "ts": ts, "value": rng.integers(-10**9, 10**9, rows)}
    dev = {k: qk.DeviceBuffer.from_numpy(np.ascontiguousarray(x)) for k, x in d.items()}
    eng = B.BatchEngine(dev["a"].ptr, dev["b"].ptr, dev["ts"].ptr, dev["value"].ptr, rows, block, 4096)
    eng.set_tuning(B.Tuning(tile, 2048, 1, graph))
    nblk = -(-rows // block)
    qs = [B.Query(0, nblk, int(I64.min), int(I64.max), 100), B.Query(0, nblk, 5, 5, 7), B.Query(0, nblk, 9, 3, 3000)]
    for i in range(40):
        first = int(rng.integers(0, nblk))
        lo, hi = sorted(int(x) for x in rng.choice(ts, 2))
        qs.append(B.Query(first, int(rng.integers(1, nblk - first + 1)), lo, hi + (i & 1 and hi < I64.max),
                          [1, 2, 3, 1000, 2048, 2049, 50_000, 1 << 20][i % 8]))
    for _ in range(2):  # the second run repeats the first over the same buffers
        eng.run(qs)
        qk._abi.call("qk_device_synchronize")
        for i, q in enumerate(qs):
            want = expect(d, q, block, rows, 4096)
            got = eng.result_arrays(i)
            np.testing.assert_array_equal(got[0], want[0])
            live = want[0] > 0
            for g, w in zip(got[1:], want[1:]):
                np.testing.assert_array_equal(g[live], w[live])
        qs = qs[::-1]
    eng.close()
