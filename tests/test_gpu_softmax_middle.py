"""softmax and log_softmax over a middle dim at the sizes where the launch
shape changes: columns in units of 4 (the last one overlapping), single
columns, positions in registers and streamed."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


@pytest.mark.parametrize("log", [False, True])
@pytest.mark.parametrize("outer,length,inner", [(3, 1, 2), (5, 2, 3), (1, 16, 2), (70, 17, 3), (2, 513, 2), (1, 2049, 3),
                                                (1, 8, 4), (300, 9, 5), (3, 64, 7), (2, 65, 66), (2, 256, 33),
                                                (1, 257, 64), (2, 1024, 31), (1, 1025, 12), (1, 2600, 257)])
def test_middle_dim(hip, outer, length, inner, log):
    print("softmax middle", outer, length, inner, log, flush=True)
    r = np.random.default_rng(outer * length * inner)
    x = (2 * r.standard_normal((outer, length, inner))).astype(np.float32)
    g = r.standard_normal(x.shape).astype(np.float32)
    y = hip.softmax_fwd(hip.DeviceArray.from_numpy(x), 1, log)
    dx = hip.softmax_bwd(y, hip.DeviceArray.from_numpy(g), 1, log).numpy().astype(np.float64)
    got = y.numpy().astype(np.float64)
    x64, g64 = x.astype(np.float64), g.astype(np.float64)
    z = x64 - x64.max(1, keepdims=True)
    lse = np.log(np.exp(z).sum(1, keepdims=True))
    # a thread's chain of positive terms (at most 32 in registers, length / 128
    # streamed), 8 combining steps, exp to 2 ulp of a difference off by z * eps
    chain = max(32, length / 128) + 16
    if log:
        want = z - lse
        assert (np.abs(got - want) <= EPS * (chain + 2 * np.abs(z) + np.abs(lse) + np.abs(want))).all()
        dwant, mag = g64 - np.exp(got) * g64.sum(1, keepdims=True), np.abs(g64).sum(1, keepdims=True) * np.exp(got)
        bound = EPS * (chain * mag + np.abs(got) * mag + 2 * np.abs(g64))
    else:
        want = np.exp(z - lse)
        assert (np.abs(got - want) <= EPS * want * (chain + np.abs(z) + 4)).all()
        dot = (g64 * got).sum(1, keepdims=True)
        dwant, mag = got * (g64 - dot), got * np.abs(g64 * got).sum(1, keepdims=True)
        bound = EPS * (chain * mag + 4 * got * (np.abs(g64) + np.abs(dot)))
    assert (np.abs(dx - dwant) <= bound + 1e-37).all()


def test_masked_and_nan_columns(hip):
    """-inf among finite values gives probability 0; a column of -inf alone,
    or with a NaN or +inf, gives NaN there and only there (registers and
    streamed alike)."""
    for length in (20, 3000):
        print("softmax middle special", length, flush=True)
        x = np.random.default_rng(length).standard_normal((1, length, 6)).astype(np.float32)
        x[0, 3:9, 0] = -np.inf
        x[0, :, 1] = -np.inf
        x[0, length - 1, 2] = np.nan
        x[0, 5, 3] = np.inf
        x[0, :, 4] = np.finfo(np.float32).min
        x[0, 2, 5] = np.finfo(np.float32).max
        y = hip.softmax_fwd(hip.DeviceArray.from_numpy(x), 1, False).numpy()[0]
        assert (y[3:9, 0] == 0).all() and abs(y[:, 0].sum() - 1) < 1e-5
        assert np.isnan(y[:, 1]).all() and np.isnan(y[:, 2]).all() and np.isnan(y[5, 3])
        np.testing.assert_allclose(y[:, 4], 1.0 / length, rtol=1e-6)
        assert y[2, 5] == 1 and (np.delete(y[:, 5], 2) == 0).all()
