"""Dim reductions at the sizes where the launch shape changes: contiguous
strips a wave, a block or many blocks each, at every float alignment, and
strided strips of few outputs folded through LDS, with ragged columns."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KINDS = ["sum", "mean", "norm", "max", "min", "argmax", "argmin"]
EPS = 2.0 ** -24


def _run(hip, kind, x, shape, strides, dim, skip):
    """oxi_reduce over a view of `x` that starts `skip` floats into it."""
    out = hip.DeviceArray(shape[:dim] + shape[dim + 1:] or (1,))
    hip.call("oxi_reduce", hip.REDUCE.index(kind), x.ptr + 4 * skip, hip._i64arr(strides), hip._i64arr(shape),
             len(shape), dim, out.ptr)
    return out.numpy().reshape(shape[:dim] + shape[dim + 1:])


def _check(got, kind, x, dim, chain):
    """arg*/max/min exactly; sums within the bound of a sum whose longest
    chain of float32 additions is `chain` (a square, a division and a root
    add a rounding each)."""
    if kind in ("max", "min", "argmax", "argmin"):
        np.testing.assert_array_equal(got, getattr(np, kind)(x, axis=dim).astype(np.float32))
        return
    x64 = x.astype(np.float64)
    if kind == "norm":
        want = np.sqrt((x64 * x64).sum(dim))
        bound = want * (chain + 3) * EPS
    else:
        n = x.shape[dim] if kind == "mean" else 1
        want = x64.sum(dim) / n
        bound = np.abs(x64).sum(dim) / n * (chain + 2) * EPS
    assert (np.abs(got - want) <= bound).all(), f"{kind}: {np.abs(got - want).max()} over {bound.min()}"


# lanes' chains: len / (4 * threads) values each, then 2 + 6 + up to 15 combining steps
@pytest.mark.parametrize("skip", [0, 1, 3])
@pytest.mark.parametrize("rows,length", [(3, 32), (5, 1023), (2, 2048), (300, 2049), (7, 2051), (600, 4100),
                                         (2, 65535), (1, 65536), (3, 65537), (255, 66000), (1, 1048583)])
def test_contiguous_strips(hip, rows, length, skip):
    print("reduce strips", rows, length, skip, flush=True)
    x = np.random.default_rng(rows * length + skip).standard_normal((rows, length), dtype=np.float32)
    buf = hip.DeviceArray.from_numpy(np.concatenate([np.full(skip, np.nan, np.float32), x.ravel()]))
    for kind in KINDS:
        got = _run(hip, kind, buf, (rows, length), (length, 1), 1, skip)
        _check(got, kind, x, 1, length // (64 * 4 if length <= 2048 else 256 * 4) + 32)


@pytest.mark.parametrize("shape,dim", [((64, 16), 0), ((65, 17), 0), ((511, 4), 0), ((512, 1003), 0), ((513, 20), 0),
                                       ((1537, 2), 0), ((5, 150, 33), 1), ((3, 1025, 768), 1), ((640, 16385), 0)])
def test_strided_strips_keep_the_sequential_order(hip, shape, dim):
    """sum, mean and norm bit for bit the sequential float32 fold."""
    print("reduce columns", shape, dim, flush=True)
    from oracle import ref

    x = np.random.default_rng(sum(shape)).standard_normal(shape, dtype=np.float32)
    buf = hip.DeviceArray.from_numpy(x)
    strides = hip.row_major_strides(shape)
    for kind in KINDS:
        np.testing.assert_array_equal(_run(hip, kind, buf, shape, strides, dim, 0), ref.reduce(kind, x, dim),
                                      err_msg=kind)


@pytest.mark.parametrize("rows,length,skip", [(5, 33, 0), (3, 63, 1), (6, 64, 0), (2, 65, 0), (9, 127, 2), (4, 128, 0),
                                              (4, 128, 3), (4, 129, 0), (5, 131, 1)])
def test_short_strips(hip, rows, length, skip):
    """Both sides of the length up to which a wave's lanes read single floats."""
    test_contiguous_strips(hip, rows, length, skip)


# full: the extents the view is cut from (its strides), rows of 1 to 4 outputs
@pytest.mark.parametrize("shape,full,dim", [((70, 100, 1), (70, 100, 1), 0), ((70, 100, 1), (70, 101, 3), 1),
                                            ((65, 64, 4), (65, 64, 4), 0), ((9, 65, 2), (9, 65, 2), 1),
                                            ((3000, 64, 3), (3000, 64, 3), 1), ((3000, 64, 4), (3001, 64, 8), 1),
                                            ((2, 600, 1, 3), (2, 600, 5, 3), 1), ((700, 1, 1), (700, 2, 2), 0)])
def test_narrow_rows_of_outputs(hip, shape, full, dim):
    """Outputs that do not lie side by side, dims of size 1 and dims that
    merge: the sequential fold's bits by either strided kernel."""
    print("reduce narrow", shape, full, dim, flush=True)
    from oracle import ref

    whole = np.random.default_rng(sum(full)).standard_normal(full, dtype=np.float32)
    x = whole[tuple(slice(0, n) for n in shape)]
    buf = hip.DeviceArray.from_numpy(whole)
    strides = hip.row_major_strides(full)
    for kind in KINDS:
        np.testing.assert_array_equal(_run(hip, kind, buf, shape, strides, dim, 0),
                                      ref.reduce(kind, np.ascontiguousarray(x), dim), err_msg=kind)


@pytest.mark.parametrize("shape", [(17, 524288), (17, 524284), (9, 1024, 1, 512), (8, 524290)])
def test_one_or_four_outputs_a_thread(hip, shape):
    print("reduce many outputs", shape, flush=True)
    test_narrow_rows_of_outputs(hip, shape, shape, 0)


@pytest.mark.parametrize("rows,cols,dim", [(4, 70000, 1), (4, 700, 1), (700, 20, 0)])
def test_first_winner_and_nan_rules(hip, rows, cols, dim):
    """Ties go to the first position, a NaN counts only at position 0, strips
    of one value (the type's lowest included) and of NaN alone give 0."""
    print("reduce ties", rows, cols, dim, flush=True)
    n, m = (cols, rows) if dim == 1 else (rows, cols)
    x = np.zeros((m, n), np.float32)
    x[0, n // 2:] = 3.0
    x[1, [5, n - 1]] = np.nan
    x[1, [9, n - 3]] = 4.0
    x[2] = -np.inf
    x[3] = np.nan
    want = {"argmax": [n // 2, 9, 0, 0], "argmin": [0, 0, 0, 0], "max": [3.0, 4.0, -np.inf, -np.inf]}
    strides = (n, 1) if dim == 1 else (1, m)
    store = x if dim == 1 else np.ascontiguousarray(x.T)
    shape = (m, n)
    buf = hip.DeviceArray.from_numpy(store)
    for kind, w in want.items():
        np.testing.assert_array_equal(_run(hip, kind, buf, shape, strides, 1, 0)[:4], np.array(w, np.float32), err_msg=kind)


def test_captured_long_strip(hip):
    """A long strip under capture takes the route without a workspace: three
    replays on new inputs, each with the eager call's sum to its rounding."""
    import ctypes

    from test_gpu_graph import CAPTURE_MODE_RELAXED, _runtime

    n = 200_003
    print("reduce captured", n, flush=True)
    rt = _runtime()
    x, out, eager = hip.DeviceArray((n,)), hip.DeviceArray((1,)), hip.DeviceArray((1,))
    st, sh = hip._i64arr((1,)), hip._i64arr((n,))

    def call(o):
        hip.call("oxi_reduce", hip.REDUCE.index("sum"), x.ptr, st, sh, 1, 0, o.ptr)

    stream, graph, exe = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    hip.check(hip.lib.oxi_hip_stream(ctypes.byref(stream)))
    hip.sync()
    held = hip.memory_stats()[0]
    assert rt.hipStreamBeginCapture(stream, CAPTURE_MODE_RELAXED) == 0
    try:
        call(out)
    finally:
        rc = rt.hipStreamEndCapture(stream, ctypes.byref(graph))
    assert rc == 0 and graph.value and hip.memory_stats()[0] == held
    try:
        assert rt.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, 0) == 0
        for k in range(3):
            v = np.random.default_rng(k).standard_normal(n, dtype=np.float32)
            hip.check(hip.lib.oxi_hip_memcpy_h2d(x.ptr, v.ctypes.data, x.nbytes))
            call(eager)
            hip.sync()
            assert rt.hipGraphLaunch(exe, stream) == 0
            hip.sync()
            for o in (out, eager):
                _check(o.numpy()[0], "sum", v, 0, n // 4096 + 32)
    finally:
        if exe.value:
            rt.hipGraphExecDestroy(exe)
        rt.hipGraphDestroy(graph)


@pytest.mark.parametrize("rows,length", [(1, 65536), (1, 200_003), (3, 1_000_001), (250, 65_541)])
def test_long_strips_have_the_same_bits_without_a_workspace(hip, rows, length):
    """Under capture, and when the workspace is refused, one launch forms the
    parts of a long strip that the eager call spreads over the chip."""
    import ctypes

    from test_gpu_graph import CAPTURE_MODE_RELAXED, _runtime

    print("reduce without a workspace", rows, length, flush=True)
    rt = _runtime()
    x = np.random.default_rng(length).standard_normal((rows, length), dtype=np.float32)
    x[0, length - 7] = np.nan
    buf = hip.DeviceArray.from_numpy(x)
    st, sh = hip._i64arr((length, 1)), hip._i64arr((rows, length))
    outs = {k: hip.DeviceArray((rows,)) for k in KINDS}

    def call(kind, o):
        hip.call("oxi_reduce", hip.REDUCE.index(kind), buf.ptr, st, sh, 2, 1, o.ptr)

    want = {k: _run(hip, k, buf, (rows, length), (length, 1), 1, 0) for k in KINDS}
    for k in KINDS:
        o = hip.DeviceArray.from_numpy(np.full(rows, -1, np.float32))
        hip.lib.oxi_hip_debug_fail_alloc_after(1)
        try:
            call(k, o)
        finally:
            hip.lib.oxi_hip_debug_fail_alloc_after(0)
        np.testing.assert_array_equal(o.numpy().view(np.uint32), want[k].view(np.uint32), err_msg=k)
    stream, graph, exe = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    hip.check(hip.lib.oxi_hip_stream(ctypes.byref(stream)))
    hip.sync()
    assert rt.hipStreamBeginCapture(stream, CAPTURE_MODE_RELAXED) == 0
    try:
        for k in KINDS:
            call(k, outs[k])
    finally:
        rc = rt.hipStreamEndCapture(stream, ctypes.byref(graph))
    assert rc == 0 and graph.value
    try:
        assert rt.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, 0) == 0
        for replay in range(3):
            for k in KINDS:
                hip.call("oxi_fill", outs[k].ptr, rows, -1.0)
            hip.sync()
            assert rt.hipGraphLaunch(exe, stream) == 0
            hip.sync()
            for k in KINDS:
                np.testing.assert_array_equal(outs[k].numpy().view(np.uint32), want[k].view(np.uint32),
                                              err_msg=f"{k}, replay {replay}")
    finally:
        if exe.value:
            rt.hipGraphExecDestroy(exe)
        rt.hipGraphDestroy(graph)


def test_more_long_strips_than_a_grid_of_blocks_holds(hip):
    """2^24 and a few strips of one broadcast row: 256 threads each would be a
    grid of more than 2^32 threads."""
    n, length = 2 ** 24 + 5, 2051
    print("reduce many strips", n, length, flush=True)
    x = np.random.default_rng(1).integers(-8, 9, length).astype(np.float32)  # sums are exact in any order
    buf = hip.DeviceArray.from_numpy(x)
    got = _run(hip, "sum", buf, (n, length), (0, 1), 1, 0)
    assert (got == x.sum(dtype=np.float64)).all()
