"""Rows whose length is not a multiple of 4, or which start at any float
alignment, through the kernels that read them as float4s."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def _at(hip, a, skip):
    """`a` on the device, `skip` floats past a 16-byte boundary (the rest NaN): (buffer, address)."""
    b = hip.DeviceArray.from_numpy(np.concatenate([np.full(skip, np.nan, np.float32), a.ravel(),
                                                   np.full(4, np.nan, np.float32)]))
    return b, b.ptr + 4 * skip


def _rows_back(buf, shape, skip):
    """The rows written, after checking that nothing around them was."""
    flat = buf.numpy()
    n = int(np.prod(shape))
    assert np.isnan(flat[:skip]).all() and np.isnan(flat[skip + n:]).all(), "written outside the rows"
    return flat[skip:skip + n].reshape(shape)


@pytest.mark.parametrize("n,c", [(3, 1), (5, 2), (4, 3), (7, 5), (6, 1001), (3, 4099), (2, 16385), (600, 18001),
                                 (3, 50257), (2, 65538)])
@pytest.mark.parametrize("xs,ds", [(0, 0), (1, 1), (2, 3)])
def test_cross_entropy(hip, n, c, xs, ds):
    """Loss, lse and gradient against float64; the sums' longest float32 chain
    is c / 1024 or, up to 16384 classes, c / 256 values a thread, and exp is
    good to 2 ulp."""
    print("cross-entropy rows", n, c, xs, ds, flush=True)
    r = np.random.default_rng(n * c + xs)
    x = (2 * r.standard_normal((n, c))).astype(np.float32)
    t = r.integers(0, c, n)
    t[0], t[-1] = 0, c - 1
    xb, xp = _at(hip, x, xs)
    db, dp = _at(hip, np.full((n, c), np.nan, np.float32), ds)
    tb = hip.DeviceArray.from_numpy(t.astype(np.int64))
    loss, lse = hip.DeviceArray((1,)), hip.DeviceArray((n,))
    one = hip.DeviceArray.from_numpy(np.ones(1, np.float32))
    hip.call("oxi_cross_entropy_fwd", xp, tb.ptr, loss.ptr, lse.ptr, n, c)
    hip.call("oxi_cross_entropy_bwd", xp, tb.ptr, lse.ptr, one.ptr, dp, n, c)
    x64 = x.astype(np.float64)
    m = x64.max(1, keepdims=True)
    want = (m + np.log(np.exp(x64 - m).sum(1, keepdims=True)))
    tol = EPS * (c / 256 + 48)
    got = lse.numpy().astype(np.float64)
    assert (np.abs(got - want[:, 0]) <= tol * (1 + np.abs(want[:, 0]))).all()
    picked = x64[np.arange(n), t] - want[:, 0]
    assert abs(float(loss.numpy()[0]) + picked.mean()) <= tol * (1 + np.abs(want).max() + np.abs(x64).max())
    # the gradient from the lse the forward gave: a subtraction (of values up
    # to |x| + |lse|), an exponential and two products
    p = np.exp(x64 - got[:, None])
    d = p.copy()
    d[np.arange(n), t] -= 1.0
    bound = EPS / n * (p * (np.abs(x64) + np.abs(got[:, None]) + 8) + np.abs(d) * 4)
    assert (np.abs(_rows_back(db, (n, c), ds) - d / n) <= bound).all()
