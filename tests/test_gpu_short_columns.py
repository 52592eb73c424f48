"""Columns shorter than a line, a line long and a key longer, through the drivers, plans and
join-aggregate strategies of the kinds that read the column by lines; the type's largest key is
found only where the column holds it."""
import numpy as np
import pytest

from gpujoin_amd import _lib

pytestmark = pytest.mark.gpu

KINDS = [("btree", {"btree_node_bytes": 64}), ("btree", {}), ("btree", {"btree_node_bytes": 256}), ("radix_spline", {}),
         ("learned_plr", {"learned_layout": 1}), ("learned_mlp", {"learned_layout": 1, "mlp_steps": 5})]
IDS = [k + "".join(f"-{v}" for v in p.values()) for k, p in KINDS]


def _column(n, dt, top):
    rng = np.random.default_rng(n)
    keys = np.cumsum(rng.integers(1, 3, n)).astype(dt) + dt(5)
    if top:
        keys[-1] = np.iinfo(dt).max
    return keys


@pytest.mark.parametrize("kind,prm", KINDS, ids=IDS)
@pytest.mark.parametrize("dt", [np.uint32, np.uint64])
@pytest.mark.parametrize("n", [1, 2, 7, 15, 16, 17, 31, 32, 33, 63, 64, 65])
@pytest.mark.parametrize("top", [False, True])
def test_lookup(gj, orc, gpu, kind, prm, dt, n, top):
    keys = _column(n, dt, top)
    print(f"[case] {kind} {prm} {dt.__name__} n={n} top={top}", flush=True)
    probes = np.concatenate([np.arange(0, 5 + 2 * n + 40, dtype=dt), np.repeat(np.array([np.iinfo(dt).max], dtype=dt), 3)])
    probes = np.random.default_rng(1).permutation(np.tile(probes, 40))
    want = orc.lookup_lower_bound(keys, probes)
    dp, out = gj.DeviceArray.from_numpy(probes), gj.DeviceArray(probes.size, np.uint32)
    idx = gj.Index(kind, gj.DeviceArray.from_numpy(keys), host_column=keys, params=gj.index_params(**prm))
    for approach, kw in (("plain", {}), ("bws", {}), ("partitioning", {"radix_bits": 3})):
        out.fill(0x5A)
        idx.lookup(dp, out, approach=approach, **kw)
        gj.synchronize()
        assert np.array_equal(out.numpy(), want), approach
    for mode in (_lib.BATCH_LAUNCH, _lib.BATCH_GRAPH, _lib.BATCH_PERSISTENT):
        half = probes.size // 2
        parts = [(0, half), (half, probes.size - half)]
        plan = gj.LookupPlan(idx, [(dp.offset(at), out.offset(at), z) for at, z in parts], mode)
        for _ in range(2):
            out.fill(0x5A)
            plan.run()
            gj.synchronize()
            assert np.array_equal(out.numpy(), want), mode
        plan.close()
    idx.close()


@pytest.mark.parametrize("kind,prm", KINDS, ids=IDS)
@pytest.mark.parametrize("dim", [1, 15, 31, 32, 63, 64])
def test_aggregate(gj, orc, gpu, kind, prm, dim):
    key, flag = gj.gen_dimension(dim, 5)
    skey, sflag = gj.sort_dimension(key, flag)
    fact = gj.gen_fact(20_003, dim + dim // 7 + 1, 2557, 90000, 10500000, 10, 6)
    idx = gj.Index(kind, gj.DeviceArray.from_numpy(skey), host_column=skey, params=gj.index_params(**prm))
    d = [gj.DeviceArray.from_numpy(a) for a in fact]
    dflag, res = gj.DeviceArray.from_numpy(sflag), gj.DeviceArray(4, np.int64)
    want = orc.join_aggregate(skey, sflag, *fact, 100, 900)
    for strategy in ("lane_refill", "plain", "partitioned", "sorted", "lookup_first"):
        res.fill(0)
        gj.join_aggregate(idx, *d, dflag, 100, 900, res, strategy=strategy)
        gj.synchronize()
        assert tuple(int(v) for v in res.numpy()[:3]) == want, strategy
    idx.close()
