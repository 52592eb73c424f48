"""The quad line search (four lanes per 128-byte line) at the edges of its lines: columns of
less than a line, of whole lines and of a line and a bit, with the largest representable
key (the fill value of partial lines) as a build key and as an absent probe."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KINDS = [("btree", {"btree_node_bytes": 64}), ("btree", {"btree_node_bytes": 128}), ("btree", {"btree_node_bytes": 256}),
         ("radix_spline", {}), ("learned_plr", {"learned_layout": 1}), ("learned_plr", {"learned_layout": 2}),
         ("learned_mlp", {"learned_layout": 1, "mlp_steps": 5}), ("hash", {})]


@pytest.mark.parametrize("kind,prm", KINDS, ids=lambda v: v if isinstance(v, str) else "-".join(map(str, v.values())))
@pytest.mark.parametrize("key_bytes", [4, 8])
@pytest.mark.parametrize("with_max", [False, True])
def test_line_edges(gj, orc, gpu, kind, prm, key_bytes, with_max):
    dt = np.uint32 if key_bytes == 4 else np.uint64
    top = np.iinfo(dt).max
    if kind == "hash" and with_max and key_bytes == 8:
        pytest.skip("the empty-slot marker cannot be stored")
    for n in (1, 2, 15, 16, 17, 31, 32, 33, 63, 65, 257, 4096, 4111):
        print(kind, prm, key_bytes, "n", n, flush=True)
        rng = np.random.default_rng(n)
        # small steps: several keys per model unit, so windows and walks cross lines
        keys = np.cumsum(rng.integers(1, 5, n)).astype(dt)
        if with_max:
            keys[-1] = top
        around = np.concatenate([keys, keys - dt(1), keys + dt(1), np.array([0, 1, top, top - 1], dtype=dt)])
        probes = rng.permutation(np.concatenate([around, rng.choice(keys, 301)]))
        want = orc.lookup_lower_bound(keys, probes)
        col, dp = gj.DeviceArray.from_numpy(keys), gj.DeviceArray.from_numpy(probes)
        out = gj.DeviceArray(probes.size, np.uint32)
        idx = gj.Index(kind, col, host_column=keys, params=gj.index_params(**prm))
        for approach in ("plain", "bws", "partitioning"):
            out.fill(0x5A)
            idx.lookup(dp, out, approach=approach)
            gj.synchronize()
            got = out.numpy()
            bad = np.flatnonzero(got != want)
            assert bad.size == 0, (n, approach, probes[bad[:4]], got[bad[:4]], want[bad[:4]])
        idx.close()


@pytest.mark.parametrize("m", [1, 63, 64, 65, 255, 256, 257, 100_003])
@pytest.mark.parametrize("grid", [0, 1, 7])
def test_grid_covers_input(gj, orc, gpu, m, grid):
    """One step per wave by default, a strided walk with the caller's grid: every probe answered once."""
    keys = gj.gen_build_keys(50_021, 8, 1, 63, 3)
    probes, _ = gj.gen_probes(keys, m, 0, 1.0, 0.2, 63, 4)
    want = orc.lookup_lower_bound(keys, probes)
    col, dp = gj.DeviceArray.from_numpy(keys), gj.DeviceArray.from_numpy(probes)
    out = gj.DeviceArray(m, np.uint32)
    for kind in ("btree", "binary_search", "learned_plr"):
        idx = gj.Index(kind, col, host_column=keys)
        for approach in ("plain", "bws", "partitioning"):
            out.fill(0x5A)
            idx.lookup(dp, out, approach=approach, grid_blocks=grid)
            gj.synchronize()
            assert np.array_equal(out.numpy(), want), (kind, approach)
        idx.close()
