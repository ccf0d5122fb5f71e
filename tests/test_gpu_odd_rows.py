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


@pytest.mark.parametrize("n,c", [(70, 33), (7, 255), (7, 256), (7, 257), (5, 319), (5, 320), (5, 321), (70000, 6)])
@pytest.mark.parametrize("xs,ds", [(0, 0), (1, 3)])
def test_cross_entropy_short_rows(hip, n, c, xs, ds):
    """Both sides of the lengths where a row goes from a float a thread to
    float4s, in the forward (320) and in the gradient (256)."""
    test_cross_entropy(hip, n, c, xs, ds)


@pytest.mark.parametrize("layer,mode", [(True, "exact"), (True, "ref"), (False, "exact"), (False, "ref")])
@pytest.mark.parametrize("rows,H,skip", [(5, 1, 0), (5, 3, 1), (3, 4, 1), (70, 5, 0), (600, 7, 3), (20, 255, 2), (700, 513, 0),
                                         (17, 769, 1), (300, 1023, 0), (40, 1026, 2), (3, 2050, 0), (300, 4097, 1),
                                         (2, 8192, 2), (4, 8193, 0), (270, 12288, 0), (2, 12288, 1), (3, 16383, 0),
                                         (2, 16385, 0)])
def test_norms(hip, rows, H, skip, layer, mode):
    """Forward and VJP against float64 formed from the float32 statistics; a
    row sum's chain is at most 16 values a thread (H / 256 in the loop kernel)
    and 24 combining steps, a column's ceil(rows / 64) values."""
    print("norm rows", rows, H, skip, layer, mode, flush=True)
    r = np.random.default_rng(rows * H + skip)
    x = (r.standard_normal((rows, H)) + 0.3).astype(np.float32)
    g = r.standard_normal((rows, H)).astype(np.float32)
    w = (1 + 0.1 * r.standard_normal(H)).astype(np.float32)
    b = (0.1 * r.standard_normal(H)).astype(np.float32)
    nan = np.full((rows, H), np.nan, np.float32)
    (xb, xp), (gb, gp), (yb, yp), (db, dp) = (_at(hip, a, skip) for a in (x, g, nan, nan))
    (wb, wp), (bb, bp), (dwb, dwp), (dbb, dbp) = (_at(hip, a, skip) for a in (w, b, nan[0], nan[0]))
    mean, rstd = hip.DeviceArray((rows,)), hip.DeviceArray((rows,))
    m = hip.NORM_VJP[mode]
    if layer:
        hip.call("oxi_layer_norm_fwd", xp, wp, bp, yp, mean.ptr, rstd.ptr, rows, H, 1e-5)
        hip.call("oxi_layer_norm_bwd", xp, wp, mean.ptr, rstd.ptr, gp, dp, dwp, dbp, rows, H, m)
    else:
        hip.call("oxi_rms_norm_fwd", xp, wp, yp, rstd.ptr, rows, H, 1e-5)
        hip.call("oxi_rms_norm_bwd", xp, wp, rstd.ptr, gp, dp, dwp, rows, H, m)
    x64, g64, w64 = x.astype(np.float64), g.astype(np.float64), w.astype(np.float64)
    chain = max(16, H / 256) + 24
    mu64 = x64.mean(1) if layer else np.zeros(rows)
    if layer:
        mu = mean.numpy().astype(np.float64)
        assert (np.abs(mu - mu64) <= EPS * chain * np.abs(x64).mean(1)).all()
        mu64 = mu
    xc = x64 - mu64[:, None]
    inv = rstd.numpy().astype(np.float64)
    assert (np.abs(inv * np.sqrt((xc * xc).mean(1) + 1e-5) - 1) <= EPS * (chain + 6 + np.abs(x64).max())).all()
    xh = xc * inv[:, None]
    err_xh = EPS * inv[:, None] * (np.abs(x64) + 2 * np.abs(xc))  # a difference and a product
    want = xh * w64 + (b if layer else 0)
    got = _rows_back(yb, (rows, H), skip)
    assert (np.abs(got - want) <= 2 * np.abs(w64) * err_xh + 4 * EPS * (np.abs(xh * w64) + np.abs(want))).all()
    gw = g64 * w64
    if mode == "ref":
        dx = gw * inv[:, None]
        mag = np.abs(dx)
        if layer:
            dx = dx - dx.mean(1, keepdims=True)
    else:
        dx = gw - xh * (gw * xh).mean(1, keepdims=True)
        mag = np.abs(gw) + np.abs(xh) * np.abs(gw * xh).mean(1, keepdims=True)
        if layer:
            dx = dx - gw.mean(1, keepdims=True)
            mag = mag + np.abs(gw).mean(1, keepdims=True)
        dx, mag = dx * inv[:, None], mag * inv[:, None]
    got = _rows_back(db, (rows, H), skip)
    slack = inv[:, None] * (err_xh * np.abs(gw * xh).mean(1, keepdims=True)
                            + np.abs(xh) * (err_xh * np.abs(gw)).mean(1, keepdims=True))
    assert (np.abs(got - dx) <= EPS * chain * (mag + mag.mean(1, keepdims=True)) + slack).all()
    cols = rows / 64 + 20
    got = _rows_back(dwb, (H,), skip)
    assert (np.abs(got - (g64 * xh).sum(0)) <= EPS * cols * np.abs(g64 * xh).sum(0) + (np.abs(g64) * err_xh).sum(0)).all()
    if layer:
        got = _rows_back(dbb, (H,), skip)
        assert (np.abs(got - g64.sum(0)) <= EPS * cols * np.abs(g64).sum(0)).all()
