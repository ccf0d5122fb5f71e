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
