"""Surrogate inference on more rows than one launch's threads can count
(2^32 in a grid dimension): the rows around every launch's border and at both
ends equal those of a small call bit for bit (a row's result does not depend on
the call it is in)."""
import numpy as np
import pytest

import mumfim_amd as m

pytestmark = pytest.mark.gpu

CHUNK = 1 << 21  # rows; the input repeats them


def rows(dev, first, count):
    """Rows [first, first + count) of a device array."""
    width = dev.shape[1]
    out = np.empty((count, width), dev.dtype)
    step = width * dev.dtype.itemsize
    m.check(m.lib().mf_memcpy_to_host(out.ctypes.data, dev.ptr + first * step, count * step))
    return out


# 2^32 threads are 2^23 workgroups of 512, of 16 rows with a Jacobian and 64 without
@pytest.mark.parametrize("jacobian,n", [(True, (1 << 27) + 33), (False, (1 << 29) + 33)])
def test_more_rows_than_one_launch_counts(jacobian, n):
    print(f"case: {n} rows, jacobian {jacobian}", flush=True)
    mlp = m.SurrogateMLP(1, 7)
    x = np.random.default_rng(4).normal(size=(CHUNK, 10)).astype(np.float32)
    X, Y = m.DeviceArray((n, 10), np.float32), m.DeviceArray((n, 6), np.float32)
    J = m.DeviceArray((n, 36), np.float32) if jacobian else None
    for r in range(0, n, CHUNK):
        c = min(CHUNK, n - r)
        m.check(m.lib().mf_memcpy_to_device(X.ptr + 40 * r, x.ctypes.data, 40 * c))
    m.check(m.lib().mf_mlp_predict_device(mlp.h, -1, X.ptr, n, Y.ptr, J.ptr if J else None, None))
    for mid in [0] + [k << 25 for k in range(1, (n >> 25) + 1)] + [n]:
        a, b = max(0, mid - 70), min(n, mid + 70)
        ref = mlp.predict(x[np.arange(a, b) % CHUNK], jacobian=jacobian)
        np.testing.assert_array_equal(rows(Y, a, b - a), ref[0])
        if jacobian:
            np.testing.assert_array_equal(rows(J, a, b - a).reshape(-1, 6, 6),
                                          np.asarray(ref[2]).reshape(-1, 6, 6))
