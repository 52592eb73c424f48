"""The column's partial last line: probes that are all in it, that reach it from the line
before and that are sent back from it, for every kind that reads column lines, and a
last bucket of binary search that holds the partial line alone or behind whole ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KINDS = [("btree", {"btree_node_bytes": 64}), ("btree", {}), ("btree", {"btree_node_bytes": 256}), ("radix_spline", {}),
         ("learned_plr", {"learned_layout": 1}), ("learned_mlp", {"learned_layout": 1, "mlp_steps": 5}),
         ("binary_search", {})]


@pytest.mark.parametrize("kind,prm", KINDS, ids=lambda v: v if isinstance(v, str) else "-".join(map(str, v.values())))
@pytest.mark.parametrize("dt", [np.uint32, np.uint64])
@pytest.mark.parametrize("rest", [1, 2, 15, 17, 31])
@pytest.mark.parametrize("base", [0, 32, 4096, 1 << 18])
def test_last_line(gj, orc, gpu, kind, prm, dt, rest, base):
    n = base + rest
    print(f"[case] {kind} {prm} {dt.__name__} n={n}", flush=True)
    rng = np.random.default_rng(n)
    keys = np.cumsum(rng.integers(1, 9, n)).astype(dt)
    keys[-min(n, 70):] += dt(40)  # a jump that the models' windows straddle
    end = keys[-min(n, 130):]
    near = np.concatenate([end, end - dt(1), end + dt(1), np.arange(keys[-1], keys[-1] + dt(99), dtype=dt)])
    top = np.array([np.iinfo(dt).max], dtype=dt)
    col = gj.DeviceArray.from_numpy(keys)
    idx = gj.Index(kind, col, host_column=keys, params=gj.index_params(**prm))
    for probes in (keys[-min(n, rest):], np.repeat(top, 64), rng.permutation(np.concatenate([near, top])),
                   rng.permutation(np.concatenate([near, rng.choice(keys, 4000)]))):
        want = orc.lookup_lower_bound(keys, probes)
        dp = gj.DeviceArray.from_numpy(probes)
        out = gj.DeviceArray(probes.size, np.uint32)
        for approach, kw in (("plain", {}), ("bws", {}), ("partitioning", {"radix_bits": 4})):
            out.fill(0x5A)
            idx.lookup(dp, out, approach=approach, **kw)
            gj.synchronize()
            assert np.array_equal(out.numpy(), want), approach
    idx.close()
