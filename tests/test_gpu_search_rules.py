"""Binary search on both sides of the rules that choose between halving and reading lines:
join-aggregate buckets of 512 and 513 keys, batch plans over buckets of 128 and 129 keys with
batches on both sides of the halvings bound; partitions of 1024 keys and a few more."""
import numpy as np
import pytest

from gpujoin_amd import _lib

pytestmark = pytest.mark.gpu


def _column(n, dt, rng):
    return np.cumsum(rng.integers(1, 5, n)).astype(dt)


@pytest.mark.parametrize("dt", [np.uint32, np.uint64])
@pytest.mark.parametrize("bits", [1, 4, 8])
@pytest.mark.parametrize("extra", [0, 1, 17])
def test_partitioned(gj, orc, gpu, dt, bits, extra):
    rng = np.random.default_rng(bits)
    keys = _column((1024 << bits) + (extra << bits), dt, rng)
    probes = np.concatenate([rng.choice(keys, 30_000), rng.choice(keys, 3_000) + dt(1), keys[-40:]])
    want = orc.lookup_lower_bound(keys, probes)
    dp = gj.DeviceArray.from_numpy(probes)
    out = gj.DeviceArray(probes.size, np.uint32)
    idx = gj.Index("binary_search", gj.DeviceArray.from_numpy(keys))
    for window in (2047, 2048, 10_000, 1 << 20):
        out.fill(0x5A)
        idx.lookup(dp, out, params=gj.lookup_params("partitioning", radix_bits=bits, window=window))
        gj.synchronize()
        assert np.array_equal(out.numpy(), want), window
    idx.close()


@pytest.mark.parametrize("dim", [1 << 20, (1 << 20) + 2048])
@pytest.mark.parametrize("strategy", ["lane_refill", "plain", "partitioned", "sorted", "lookup_first"])
def test_aggregate(gj, orc, gpu, dim, strategy):
    key, flag = gj.gen_dimension(dim, 5)
    skey, sflag = gj.sort_dimension(key, flag)
    fact = gj.gen_fact(200_003, dim + dim // 7, 2557, 90000, 10500000, 10, 6)
    idx = gj.Index("binary_search", gj.DeviceArray.from_numpy(skey))
    res = gj.DeviceArray(4, np.int64)
    res.fill(0)
    d = [gj.DeviceArray.from_numpy(a) for a in fact]
    dflag = gj.DeviceArray.from_numpy(sflag)
    gj.join_aggregate(idx, *d, dflag, 100, 900, res, strategy=strategy)
    gj.synchronize()
    assert tuple(int(v) for v in res.numpy()[:3]) == orc.join_aggregate(skey, sflag, *fact, 100, 900)
    idx.close()


@pytest.mark.parametrize("dt", [np.uint32, np.uint64])
@pytest.mark.parametrize("n", [2048 * 128, 2048 * 128 + 1])
@pytest.mark.parametrize("mode", [_lib.BATCH_LAUNCH, _lib.BATCH_GRAPH, _lib.BATCH_PERSISTENT])
def test_plans(gj, orc, gpu, dt, n, mode):
    rng = np.random.default_rng(n)
    keys = _column(n, dt, rng)
    sizes = [1, 64, 1000, 163_839, 163_841, 200_003]  # 8 halvings a probe: the bound is 163840
    probes = rng.choice(keys, sum(sizes))
    probes[::9] += dt(1)
    want = orc.lookup_lower_bound(keys, probes)
    dp, out = gj.DeviceArray.from_numpy(probes), gj.DeviceArray(probes.size, np.uint32)
    idx = gj.Index("binary_search", gj.DeviceArray.from_numpy(keys))
    batches, at = [], 0
    for z in sizes:
        batches.append((dp.offset(at), out.offset(at), z))
        at += z
    plan = gj.LookupPlan(idx, batches, mode)
    for _ in range(3):
        out.fill(0x5A)
        plan.run()
        gj.synchronize()
        assert np.array_equal(out.numpy(), want)
    plan.close()
    idx.close()
