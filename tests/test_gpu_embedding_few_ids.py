"""The embedding VJP at the sizes where its sort changes: ids ranked in one
launch, radix-sorted on the library stream or on the second stream."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000, 4095, 4096, 4097, 32768, 32769])
@pytest.mark.parametrize("V,D,hot", [(1, 5, 0.0), (300, 8, 0.5), (50257, 12, 0.1), (200000, 1, 0.9)])
def test_exact_sums(hip, n, V, D, hot):
    """Gradients that are small whole numbers sum exactly in any order; `hot`
    of the ids are one key; negative ids count from the end. Through the plan
    (applied twice) and in one call."""
    print("embedding few ids", n, V, D, hot, flush=True)
    r = np.random.default_rng(n + V)
    ids = r.integers(-V, V, n)
    ids[r.random(n) < hot] = V // 2
    g = r.integers(-8, 9, (n, D)).astype(np.float32)
    want = np.zeros((V, D))
    np.add.at(want, np.where(ids < 0, ids + V, ids), g)
    di, dg = hip.DeviceArray.from_numpy(ids.astype(np.int64)), hip.DeviceArray.from_numpy(g)
    plan = hip.BwdPlan(di, V)
    for got in (plan.apply(dg, (V, D), 0), plan.apply(dg, (V, D), 0), hip.index_select_bwd(dg, (V, D), 0, di)):
        np.testing.assert_array_equal(got.numpy(), want)
    plan.free()


@pytest.mark.parametrize("n,V", [(4800, 300), (4801, 300), (32768, 2048), (32768, 2047), (32768, 70000), (32769, 70000)])
def test_passes_counted_by_the_scatter_or_on_their_own(hip, n, V):
    """Both sides of the sizes where a pass's counts come from the scatter
    before it (two and three passes)."""
    test_exact_sums(hip, n, V, 3, 0.3)


@pytest.mark.parametrize("n", [1, 4096])
def test_few_ids_of_many_rows(hip, n):
    """The one-launch sort's 64 blocks write the presence flags of 46876 rows
    each, 1024 at a time, the last block's share cut."""
    test_exact_sums(hip, n, 3_000_001, 1, 0.3)


@pytest.mark.parametrize("n", [5, 4096])
def test_sequential_order_and_guard(hip, n):
    """Short runs add their rows in position order; an id out of range is
    reported and adds to no row."""
    print("embedding order", n, flush=True)
    r = np.random.default_rng(n)
    V, D = n, 6
    ids = r.permutation(np.arange(n) // 2 * 2)  # pairs
    g = r.standard_normal((n, D)).astype(np.float32)
    want = np.zeros((V, D), np.float32)
    for k, i in enumerate(ids):
        want[i] += g[k]
    di, dg = hip.DeviceArray.from_numpy(ids.astype(np.int64)), hip.DeviceArray.from_numpy(g)
    np.testing.assert_array_equal(hip.index_select_bwd(dg, (V, D), 0, di).numpy(), want)
    bad = ids.copy()
    bad[3] = V
    want[ids[3]] = np.float32(0)
    for k in np.flatnonzero(bad == ids[3]):
        want[ids[3]] += g[k]
    got = hip.index_select_bwd(dg, (V, D), 0, hip.DeviceArray.from_numpy(bad.astype(np.int64)))
    with pytest.raises(RuntimeError, match="outside its valid range"):
        hip.sync()
    np.testing.assert_array_equal(got.numpy(), want)
    hip.sync()


@pytest.mark.parametrize("n", [65537, 524289, 2_100_000])
@pytest.mark.parametrize("V,hot", [(255, 0.3), (256, 1.0), (70000, 0.3)])
def test_passes_and_tiles(hip, n, V, hot):
    """Sorts of one, two and three passes, each counting for the next, over
    tiles of 2048 and 8192 ids and over more tiles than a block scans itself."""
    print("embedding passes", n, V, hot, flush=True)
    r = np.random.default_rng(n + V)
    ids = r.integers(0, V, n)
    ids[r.random(n) < hot] = V - 1
    g = r.integers(-3, 4, (n, 1)).astype(np.float32)
    want = np.bincount(ids, g[:, 0], V)[:, None]
    got = hip.index_select_bwd(hip.DeviceArray.from_numpy(g), (V, 1), 0, hip.DeviceArray.from_numpy(ids.astype(np.int64)))
    np.testing.assert_array_equal(got.numpy(), want)
