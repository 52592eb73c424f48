"""The partitioned driver over windows swept together (no more probes in a window than the
column has lines) and one after the other: few and many windows, a short last one, skewed
and sorted probes, whose windows differ, and one and two passes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["btree", "learned_plr", "binary_search", "hash"])
@pytest.mark.parametrize("dt", [np.uint32, np.uint64])
@pytest.mark.parametrize("order", ["uniform", "sorted", "hot"])
def test_windows(gj, orc, gpu, kind, dt, order):
    rng = np.random.default_rng(7)
    n = 300_032
    keys = np.unique(rng.integers(0, np.iinfo(dt).max, n + n // 8, dtype=dt))[:n]
    m = 100_003
    probes = rng.choice(keys, m)
    if order == "sorted":
        probes.sort()
    elif order == "hot":
        probes[rng.random(m) < 0.9] = keys[n // 3]
    probes[::11] += dt(1)
    want = orc.lookup_lower_bound(keys, probes)
    col, dp = gj.DeviceArray.from_numpy(keys), gj.DeviceArray.from_numpy(probes)
    out = gj.DeviceArray(m, np.uint32)
    idx = gj.Index(kind, col, host_column=keys)
    lines = n * keys.itemsize // 128
    for window in (1, 100, 4096, lines, lines + 1, 50_000, m, 1 << 24):
        if window == 1:
            part = 65  # as many windows as probes
        else:
            part = m
        for bits, passes in ((1, 1), (6, 1), (9, 2)):
            for grid in (0, 3):
                out.fill(0x5A)
                idx.lookup(dp, out, m=part, params=gj.lookup_params("partitioning", radix_bits=bits, passes=passes, window=window,
                                                                    grid_blocks=grid))
                gj.synchronize()
                assert np.array_equal(out.numpy()[:part], want[:part]), (window, bits, passes, grid)
    assert idx.stats()["dropped_tuples"] == 0
    idx.close()
