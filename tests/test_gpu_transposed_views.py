"""Elementwise calls over transposed operands whose extents, strides or
addresses are not multiples of 4 floats, at the edges of the 32 x 32 tiles and
of the 4 x 4 blocks in them (the last block of a dim repeats elements)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dev(hip, a, skip):
    b = hip.DeviceArray.from_numpy(np.concatenate([np.full(skip, np.nan, np.float32), a.ravel()]))
    return b, b.ptr + 4 * skip


@pytest.mark.parametrize("B,J,D,skip", [(1, 3, 40, 0), (2, 4, 5, 0), (3, 5, 4, 1), (2, 7, 33, 0), (1, 31, 34, 2),
                                        (2, 33, 31, 0), (3, 64, 65, 1), (2, 65, 64, 0), (2, 32, 96, 3), (1, 129, 1023, 0),
                                        (5, 1023, 30, 0)])
def test_bit_exact(hip, B, J, D, skip):
    """y (B, J, D) from operands stored (B, D, J), (B, J, D) or broadcast:
    copies and sums bit for bit, nothing outside written."""
    print("transposed", B, J, D, skip, flush=True)
    r = np.random.default_rng(B * J * D + skip)
    t = r.standard_normal((B, D, J)).astype(np.float32)  # stored transposed
    u = r.standard_normal((B, J, D)).astype(np.float32)
    col = r.standard_normal((B, J, 1)).astype(np.float32)
    (tb, tp), (ub, up), (cb, cp) = (_dev(hip, a, skip) for a in (t, u, col))
    arr = hip._i64arr
    shape, rm = arr((B, J, D)), arr((J * D, D, 1))
    tv, cv = arr((D * J, 1, J)), arr((J, 1, 0))
    n = B * J * D
    add = hip.BINARY.index("add")
    want_t = t.transpose(0, 2, 1)

    def run(call, want, what):
        out = hip.DeviceArray.from_numpy(np.full(n + skip + 8, np.nan, np.float32))
        call(out.ptr + 4 * skip)
        flat = out.numpy()
        np.testing.assert_array_equal(flat[skip:skip + n].reshape(B, J, D), want, err_msg=what)
        assert np.isnan(flat[:skip]).all() and np.isnan(flat[skip + n:]).all(), what

    run(lambda o: hip.call("oxi_unary", hip.UNARY.index("identity"), tp, tv, o, rm, shape, 3), want_t, "copy")
    run(lambda o: hip.call("oxi_binary", add, tp, tv, up, rm, o, rm, shape, 3), want_t + u, "t + u")
    run(lambda o: hip.call("oxi_binary", add, up, rm, tp, tv, o, rm, shape, 3), u + want_t, "u + t")
    run(lambda o: hip.call("oxi_binary", add, tp, tv, tp, tv, o, rm, shape, 3), want_t + want_t, "t + t")
    run(lambda o: hip.call("oxi_binary", add, tp, tv, cp, cv, o, rm, shape, 3), want_t + col, "t + column")


@pytest.mark.parametrize("B,J,D", [(3, 4, 5), (100, 7, 7), (1030, 7, 7), (2, 11, 11), (130, 11, 9), (40, 11, 4), (2, 5, 1001),
                                   (2100, 9, 5)])
def test_long_operations(hip, B, J, D):
    """Both sides of the sizes where long operations leave the registers for
    LDS tiles: the bits of the same call on a contiguous copy."""
    print("transposed, long", B, J, D, flush=True)
    r = np.random.default_rng(B * J * D)
    t, u = (r.uniform(0.1, 3, s).astype(np.float32) for s in ((B, D, J), (B, J, D)))
    flat = hip.DeviceArray.from_numpy(np.ascontiguousarray(t.transpose(0, 2, 1)))
    td, ud, shape, tv = hip.DeviceArray.from_numpy(t), hip.DeviceArray.from_numpy(u), (B, J, D), (D * J, 1, J)
    rm = hip.row_major_strides(shape)
    for what, got, want in (
            ("tanh", hip.unary("tanh", td, x_strides=tv, shape=shape), hip.unary("tanh", flat)),
            ("silu", hip.silu_fwd(td, x_strides=tv, shape=shape), hip.silu_fwd(flat)),
            ("silu vjp", hip.silu_bwd(td, ud, x_strides=tv, g_strides=rm, shape=shape), hip.silu_bwd(flat, ud)),
            ("gelu vjp", hip.gelu_bwd(td, ud, "tanh", x_strides=tv, g_strides=rm, shape=shape), hip.gelu_bwd(flat, ud, "tanh")),
            ("pow", hip.binary("pow", td, ud, tv, rm, shape), hip.binary("pow", flat, ud, rm, rm, shape))):
        np.testing.assert_array_equal(got.numpy().view(np.uint32), want.numpy().view(np.uint32), err_msg=what)
