"""The blockwise-sorting driver over a column, or index structures, in host memory, where a
wave looks up a quarter or half as many probes at a time: tiles of one probe, of less than
a wave's share, of a remainder, whole ones, a caller's grid, and enough tiles to take fewer
lanes (more than two for each CU)."""
import numpy as np
import pytest

from gpujoin_amd import _lib

pytestmark = pytest.mark.gpu

KINDS = ["binary_search", "btree", "harmonia", "radix_spline", "learned_plr", "learned_mlp", "hash"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("dt", [np.uint32, np.uint64])
@pytest.mark.parametrize("column_in_host", [False, True])
def test_bws_over_the_host_link(gj, orc, gpu, kind, dt, column_in_host):
    rng = np.random.default_rng(11)
    keys = np.unique(rng.integers(1, np.iinfo(dt).max, 40_000, dtype=dt))
    keys = keys[:keys.size // 32 * 32]
    col = gj.HostArray.from_numpy(keys) if column_in_host else gj.DeviceArray.from_numpy(keys)
    idx = gj.Index(kind, col, host_column=keys, params=gj.index_params(placement=_lib.PLACE_HOST, mlp_steps=20))
    two_tiles = 2 * gj.device_info()["compute_units"] * 2048
    for m in (1, 63, 65, 2047, 2049, two_tiles, two_tiles + 1, two_tiles + 2063):
        probes = rng.choice(keys, m) + rng.integers(0, 2, m).astype(dt)
        dp, out = gj.DeviceArray.from_numpy(probes), gj.DeviceArray(m, np.uint32)
        for grid in (0, 3):
            out.fill(0x5A)
            idx.lookup(dp, out, approach="bws", grid_blocks=grid)
            gj.synchronize()
            assert np.array_equal(out.numpy(), orc.lookup_lower_bound(keys, probes)), (m, grid)
    idx.close()
    if column_in_host:
        col.free()
