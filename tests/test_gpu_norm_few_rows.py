"""The norm VJPs that form dw and db in the launch of dx (up to 256 rows): the
bits of the two launches that more rows take."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


SHAPES = [(1, 4), (3, 260), (16, 768), (17, 768), (255, 768), (256, 1000), (250, 1024), (16, 2048), (17, 2048),
          (256, 4096), (100, 8192), (9, 1003), (256, 513), (200, 4099), (130, 12288)]
# the folded VJPs take rows of a multiple of 4 and up to 8192 floats
CASES = [(r, h, a) for r, h in SHAPES for a in ("none", "gelu_tanh", "gelu_erf", "silu")
         if a == "none" or (h % 4 == 0 and h <= 8192)]


@pytest.mark.parametrize("rows,H,act", CASES)
@pytest.mark.parametrize("layer,mode", [(True, "ref"), (False, "exact")])
def test_same_bits_as_with_more_rows(hip, rows, H, act, layer, mode):
    """Rows with a zero gradient after the others leave dw and db as they are."""
    print("norm few rows", rows, H, act, layer, mode, flush=True)
    r = np.random.default_rng(rows * H)
    more = 600
    x = r.standard_normal((more, H)).astype(np.float32)
    g = np.zeros((more, H), np.float32)
    g[:rows] = r.standard_normal((rows, H))
    D = hip.DeviceArray.from_numpy
    w, b = D((1 + 0.1 * r.standard_normal(H)).astype(np.float32)), D(r.standard_normal(H).astype(np.float32))

    def vjp(n):
        dx, dg = D(x[:n]), D(g[:n])
        if layer:
            _, mean, rstd = hip.layer_norm_fwd(dx, w, b)
            if act == "none":
                out = hip.layer_norm_bwd(dx, w, mean, rstd, dg, mode)
            else:
                out = hip.layer_norm_act_bwd(dx, w, b, mean, rstd, dg, act, mode)
        else:
            _, rstd = hip.rms_norm_fwd(dx, w)
            if act == "none":
                out = hip.rms_norm_bwd(dx, w, rstd, dg, mode)
            else:
                out = hip.rms_norm_act_bwd(dx, w, rstd, dg, act, mode)
        return [o.numpy()[:rows] if o.shape == (n, H) else o.numpy() for o in out]

    for got, want in zip(vjp(rows), vjp(more)):
        np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("rows,H", [(128, 2552), (129, 2552), (129, 4096), (256, 4092)])
def test_tanh_gelu_rows_of_a_few_thousand(hip, rows, H):
    """Both sides of the rows where the folded tanh GELU goes back to two launches."""
    test_same_bits_as_with_more_rows(hip, rows, H, "gelu_tanh", True, "ref")


def test_only_one_of_dw_and_db(hip):
    print("norm few rows, one gradient", flush=True)
    r = np.random.default_rng(1)
    D = hip.DeviceArray.from_numpy
    x, g, w = (D(r.standard_normal(s).astype(np.float32)) for s in ((40, 768), (40, 768), (768,)))
    _, mean, rstd = hip.layer_norm_fwd(x, w, None)
    both = hip.layer_norm_bwd(x, w, mean, rstd, g)
    for need in ((True, True, False), (True, False, True), (False, True, True), (False, True, False)):
        got = hip.layer_norm_bwd(x, w, mean, rstd, g, "ref", *need)
        for k in range(3):
            if need[k]:
                np.testing.assert_array_equal(got[k].numpy().view(np.uint32), both[k].numpy().view(np.uint32))


def test_captured(hip):
    """Up to 256 rows dw and db need no workspace, so the call can be captured:
    three replays on new inputs have the eager call's bits."""
    import ctypes

    from test_gpu_graph import CAPTURE_MODE_RELAXED, _runtime

    print("norm few rows, captured", flush=True)
    rt = _runtime()
    rows, H = 256, 1003
    D = hip.DeviceArray
    x, g, dx = D((rows, H)), D((rows, H)), D((rows, H))
    w, dw, db = D.from_numpy(np.linspace(0.5, 1.5, H, dtype=np.float32)), D((H,)), D((H,))
    mean, rstd = D((rows,)), D((rows,))

    def call():
        hip.call("oxi_layer_norm_bwd", x.ptr, w.ptr, mean.ptr, rstd.ptr, g.ptr, dx.ptr, dw.ptr, db.ptr, rows, H,
                 hip.NORM_VJP["exact"])

    stream, graph, exe = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    hip.check(hip.lib.oxi_hip_stream(ctypes.byref(stream)))
    hip.sync()
    held = hip.memory_stats()[0]
    assert rt.hipStreamBeginCapture(stream, CAPTURE_MODE_RELAXED) == 0
    try:
        call()
    finally:
        rc = rt.hipStreamEndCapture(stream, ctypes.byref(graph))
    assert rc == 0 and graph.value and hip.memory_stats()[0] == held
    try:
        assert rt.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, 0) == 0
        for k in range(3):
            r = np.random.default_rng(k)
            for d, v in ((x, r.standard_normal((rows, H))), (g, r.standard_normal((rows, H))),
                         (mean, 0.1 * r.standard_normal(rows)), (rstd, r.uniform(0.5, 2, rows))):
                v = v.astype(np.float32)
                hip.check(hip.lib.oxi_hip_memcpy_h2d(d.ptr, v.ctypes.data, v.nbytes))
            call()
            want = [o.numpy().copy() for o in (dx, dw, db)]
            for o in (dx, dw, db):
                hip.call("oxi_fill", o.ptr, o.size, -1.0)
            hip.sync()
            assert rt.hipGraphLaunch(exe, stream) == 0
            hip.sync()
            for o, v in zip((dx, dw, db), want):
                np.testing.assert_array_equal(o.numpy().view(np.uint32), v.view(np.uint32))
    finally:
        if exe.value:
            rt.hipGraphExecDestroy(exe)
        rt.hipGraphDestroy(graph)
