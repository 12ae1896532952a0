"""Stable compaction at the edges of its tiles (a wavefront's words, tiles of 1024 and 4096 rows, the
sizes where the tile and the scan change), by mask and by predicates, against numpy: bit-exact."""
import numpy as np
import pytest

import qikkdb_amd as qk
from gpu_util import col
from helpers import unpack_bits

pytestmark = pytest.mark.gpu
SIZES = [1, 63, 64, 65, 1023, 1025, 4097, 262_139, (1 << 21) - 1, (1 << 21) + 1, (1 << 23) + 4097]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("keep", [0.0, 0.02, 0.5, 1.0])
def test_compact_by_mask(n, keep):
    rng = np.random.default_rng(n)
    mask = np.where(rng.random(n) < keep, rng.choice(np.array([1, 2, -1, -128], np.int8), n), 0).astype(np.int8)
    isnull = rng.random(n) < 0.4
    m = qk.DeviceBuffer.from_numpy(mask)
    rows = np.flatnonzero(mask)
    for dt in (np.int8, np.int16, np.int32, np.float64):
        v = rng.integers(-100, 100, n).astype(dt)
        buf = qk.DeviceBuffer.from_numpy(v)
        nulls = qk.DeviceBuffer.from_numpy(qk.pack_nulls(isnull))
        ob, cnt, nb = qk.GPUReconstruct.reconstructColKeep(buf, v.itemsize, m, n, nulls)
        assert cnt == rows.size
        if cnt:
            np.testing.assert_array_equal(ob.to_numpy(dt, cnt), v[rows])
            words = nb.to_numpy(np.uint64)
            np.testing.assert_array_equal(qk.unpack_nulls(words, cnt), isnull[rows])
            assert not qk.unpack_nulls(words, words.size * 64)[cnt:].any()
    for size, dt in ((4, np.int32), (8, np.int64)):
        np.testing.assert_array_equal(qk.GPUReconstruct.GenerateIndexes(m, n, size), rows.astype(dt))


def test_compact_unaligned_mask():
    rng = np.random.default_rng(5)
    n = 70_001
    mask = (rng.random(n + 3) < 0.3).astype(np.int8)
    whole = qk.DeviceBuffer.from_numpy(mask)
    for off in (1, 3):
        m = qk.DeviceBuffer(n, ptr=whole.ptr + off, owned=False)
        np.testing.assert_array_equal(qk.GPUReconstruct.GenerateIndexes(m, n), np.flatnonzero(mask[off:off + n]))


@pytest.mark.parametrize("n", [1, 65, 1025, 262_139, (1 << 21) + 1])
@pytest.mark.parametrize("form", ["two_columns", "narrow", "rest", "nan"])
def test_compact_by_predicates(n, form):
    """Predicates that fold (several on one column, columns of every width, constants of another
    type), mixed with ones that do not (!=, two columns), and a NaN constant, which drops every row."""
    rng = np.random.default_rng(n)
    i8, i32 = rng.integers(-5, 6, n).astype(np.int8), rng.integers(-50, 50, n).astype(np.int32)
    i64, f32 = rng.integers(-10**12, 10**12, n), rng.normal(0, 1, n).astype(np.float32)
    f64 = rng.normal(0, 1, n)
    f32[rng.random(n) < 0.05] = np.nan
    isnull = rng.random(n) < 0.1
    c8, c32, c64, cf, cd = col(i8), col(i32, isnull), col(i64), col(f32), col(f64)
    if form == "two_columns":
        preds = [qk.where(qk.GREATER, c64, qk.Const(-10**11, qk.LONG)), qk.where(qk.LESS, cf, qk.Const(0.25, qk.DOUBLE)),
                 qk.where(qk.LESS_EQUAL, c64, qk.Const(5e11, qk.DOUBLE))]
        want = (i64 > -10**11) & (f32.astype(np.float64) < 0.25) & (i64.astype(np.float64) <= 5e11)
    elif form == "narrow":
        preds = [qk.where(qk.GREATER_EQUAL, c8, qk.Const(-2, qk.INT8)), qk.where(qk.LESS, c32, qk.Const(10.5, qk.FLOAT)),
                 qk.where(qk.EQUAL, c8, qk.Const(3, qk.LONG))]
        want = (i8 == 3) & (i32 < 10.5) & ~isnull
    elif form == "rest":
        preds = [qk.where(qk.NOT_EQUAL, c32, qk.Const(7, qk.INT)), qk.where(qk.LESS, cd, cf), qk.where(qk.GREATER, cd, qk.Const(-1.0, qk.DOUBLE))]
        want = (i32 != 7) & ~isnull & (f64 < f32.astype(np.float64)) & (f64 > -1.0)
    else:
        preds = [qk.where(qk.GREATER, cd, qk.Const(-1.0, qk.DOUBLE)), qk.where(qk.LESS, cd, qk.Const(float("nan"), qk.DOUBLE))]
        want = np.zeros(n, bool)
    rows = np.flatnonzero(want)
    outs, cnt = qk.GPUReconstruct.WhereCompact(preds, [c8, c32, c64, cf, cd], n)
    assert cnt == rows.size
    for o, v in zip(outs, (i8, i32, i64, f32, f64)):
        np.testing.assert_array_equal(o.to_numpy(), v[rows])
    if cnt:
        np.testing.assert_array_equal(unpack_bits(outs[1].nulls.to_numpy(np.uint64), cnt), isnull[rows])
