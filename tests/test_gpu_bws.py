"""Blockwise sorting at the edges of its tiles (2048 probes), with every probe in one bin, bins
finer and coarser than the tile, no staged levels at all, and every block size it accepts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KINDS = [("binary_search", {}), ("btree", {}), ("btree", {"btree_lds_bytes": 1}), ("btree", {"btree_lds_bytes": 65536}),
         ("harmonia", {}), ("radix_spline", {}), ("radix_spline", {"rs_radix_bits": 4}), ("hash", {}),
         ("learned_plr", {"learned_layout": 1}), ("learned_plr", {"learned_layout": 2}),
         ("learned_mlp", {"learned_layout": 2, "mlp_steps": 5})]


@pytest.mark.parametrize("kind,prm", KINDS, ids=lambda v: v if isinstance(v, str) else "-".join(map(str, v.values())))
@pytest.mark.parametrize("key_bytes", [4, 8])
def test_tiles(gj, orc, gpu, kind, prm, key_bytes):
    dt = np.uint32 if key_bytes == 4 else np.uint64
    top = np.iinfo(dt).max
    for n in (32, 4096, 70_016):
        rng = np.random.default_rng(n)
        keys = np.unique(rng.integers(1, top, n + n // 8, dtype=dt))[:n]
        assert keys.size == n
        col = gj.DeviceArray.from_numpy(keys)
        idx = gj.Index(kind, col, host_column=keys, params=gj.index_params(**prm))
        for m, block in ((1, 64), (2047, 128), (2048, 192), (2049, 256), (10_000, 256)):
            for probes in (rng.choice(keys, m), np.full(m, keys[n // 2]), rng.integers(0, top, m, dtype=dt, endpoint=True)):
                dp = gj.DeviceArray.from_numpy(probes.astype(dt))
                out = gj.DeviceArray(m, np.uint32)
                out.fill(0x5A)
                idx.lookup(dp, out, params=gj.lookup_params("bws", block_size=block))
                gj.synchronize()
                assert np.array_equal(out.numpy(), orc.lookup_lower_bound(keys, probes.astype(dt))), (n, m)
        idx.close()
