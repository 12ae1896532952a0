"""The int8 filter at the tails of its lanes (4 and 8 rows) and on pointers of every alignment, against
numpy: bit-exact."""
import numpy as np
import pytest

import qikkdb_amd as qk

pytestmark = pytest.mark.gpu
OPS = {qk.GREATER: np.greater, qk.GREATER_EQUAL: np.greater_equal, qk.LESS: np.less, qk.LESS_EQUAL: np.less_equal,
       qk.EQUAL: np.equal, qk.NOT_EQUAL: np.not_equal}


@pytest.mark.parametrize("n", [1, 3, 4, 7, 9, 257, 100_003, (1 << 22) + 5, 256 * 2048 * 8 + 13])
@pytest.mark.parametrize("dt", [np.int8, np.int32, np.int64, np.float32, np.float64])
def test_filter_tails_and_alignment(n, dt):
    rng = np.random.default_rng(n)
    a, b = rng.integers(-3, 4, n + 1).astype(dt), rng.integers(-3, 4, n + 1).astype(dt)
    isnull = rng.random(n) < 0.2
    nulls = qk.DeviceBuffer.from_numpy(qk.pack_nulls(isnull))
    da, db = qk.DeviceBuffer.from_numpy(a), qk.DeviceBuffer.from_numpy(b)
    qt, size = qk._abi.TYPE_OF[np.dtype(dt)], np.dtype(dt).itemsize
    out = qk.DeviceBuffer(n + 16)
    for i, (op, f) in enumerate(OPS.items()):
        shift = i & 1  # an element off, and the mask a few bytes off
        ca = qk.DeviceColumn(qk.DeviceBuffer(n * size, ptr=da.ptr + shift * size, owned=False), qt, n)
        cb = qk.DeviceColumn(qk.DeviceBuffer(n * size, ptr=db.ptr, owned=False), qt, n)
        m = qk.DeviceBuffer(n, ptr=out.ptr + i, owned=False)
        x, y = a[shift:shift + n], b[:n]
        qk.GPUBinary.Filter(op, ca, cb, n, nulls, out=m)
        np.testing.assert_array_equal(m.to_numpy(np.int8, n), (f(x, y) & ~isnull).astype(np.int8))
        qk.GPUBinary.Filter(op, ca, qk.Const(1, qt), n, None, out=m)
        np.testing.assert_array_equal(m.to_numpy(np.int8, n), f(x, dt(1)).astype(np.int8))
        qk.GPUBinary.Filter(op, qk.Const(1, qt), cb, n, nulls, out=m)
        np.testing.assert_array_equal(m.to_numpy(np.int8, n), (f(dt(1), y) & ~isnull).astype(np.int8))
