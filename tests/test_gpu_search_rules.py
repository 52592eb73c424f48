"""Binary search on both sides of the rules that choose between halving and reading lines:
join-aggregate buckets of 512 and 513 keys, batch plans over buckets of 128 and 129 keys with
batches on both sides of the halvings bound; partitions of 1024 keys and a few more; aggregates
on both sides of the row bound."""
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


@pytest.mark.parametrize("dim", [2048 * 16, 2048 * 17, 300_000])
@pytest.mark.parametrize("strategy", ["lane_refill", "sorted", "lookup_first"])
def test_aggregate_by_rows(gj, orc, gpu, dim, strategy):
    # lane refill and sorted read lines from 5 * 2^24 halvings over their rows on: 9 or 10 a row at
    # 300000 keys, 4 or 5 at 32768; lookup-first in buckets of 17 keys
    key, flag = gj.gen_dimension(dim, 5)
    skey, sflag = gj.sort_dimension(key, flag)
    fact = gj.gen_fact(21_000_001, dim + dim // 7, 2557, 90000, 10500000, 10, 6)
    idx = gj.Index("binary_search", gj.DeviceArray.from_numpy(skey))
    d, dflag = [gj.DeviceArray.from_numpy(a) for a in fact], gj.DeviceArray.from_numpy(sflag)
    res = gj.DeviceArray(4, np.int64)
    for rows in (1_000_003, 9_000_001, 21_000_001):
        res.fill(0)
        gj.join_aggregate(idx, *d, dflag, 100, 130, res, strategy=strategy, rows=rows)
        gj.synchronize()
        want = orc.join_aggregate(skey, sflag, *[a[:rows] for a in fact], 100, 130)
        assert tuple(int(v) for v in res.numpy()[:3]) == want, rows
    idx.close()


@pytest.mark.parametrize("sizes", [[1000, 70, 30_000], [1000, 9_000_001, 5_000_003]])
@pytest.mark.parametrize("mode", [_lib.BATCH_LAUNCH, _lib.BATCH_GRAPH, _lib.BATCH_PERSISTENT])
def test_aggregate_plans(gj, orc, gpu, sizes, mode):
    dim = 300_000
    key, flag = gj.gen_dimension(dim, 5)
    skey, sflag = gj.sort_dimension(key, flag)
    fact = gj.gen_fact(sum(sizes), dim + dim // 7, 2557, 90000, 10500000, 10, 6)
    idx = gj.Index("binary_search", gj.DeviceArray.from_numpy(skey))
    d, dflag = [gj.DeviceArray.from_numpy(a) for a in fact], gj.DeviceArray.from_numpy(sflag)
    res = gj.DeviceArray(4 * len(sizes), np.int64)
    starts = np.concatenate([[0], np.cumsum(sizes)]).astype(int)
    plan = gj.AggregatePlan(idx, [tuple(a.offset(int(s)) for a in d) + (z,) for s, z in zip(starts, sizes)], dflag, 100, 130,
                            res, mode)
    for _ in range(2):
        res.fill(0x5A)
        plan.run()
        gj.synchronize()
        got = res.numpy().reshape(-1, 4)
        for i, z in enumerate(sizes):
            want = orc.join_aggregate(skey, sflag, *[a[starts[i]:starts[i] + z] for a in fact], 100, 130)
            assert tuple(int(v) for v in got[i, :3]) == want, i
    plan.close()
    idx.close()


@pytest.mark.parametrize("dt", [np.uint32, np.uint64])
@pytest.mark.parametrize("many", [2_621_439, 2_621_441])
def test_persistent_plan_by_probes(gj, orc, gpu, dt, many):
    # persistent plans read lines in smaller buckets from 5 * 2^22 halvings over all their probes
    # on: 8 a probe over the 256 keys of a bucket here
    rng = np.random.default_rng(3)
    keys = _column((1024 if dt == np.uint64 else 2048) * 256 - 5, dt, rng)
    sizes = [many - 1_000_100, 1_000_000, 100]
    probes = rng.choice(keys, many)
    probes[::9] += dt(1)
    dp, out = gj.DeviceArray.from_numpy(probes), gj.DeviceArray(many, np.uint32)
    idx = gj.Index("binary_search", gj.DeviceArray.from_numpy(keys))
    starts = np.concatenate([[0], np.cumsum(sizes)]).astype(int)
    plan = gj.LookupPlan(idx, [(dp.offset(int(s)), out.offset(int(s)), z) for s, z in zip(starts, sizes)],
                         _lib.BATCH_PERSISTENT)
    for _ in range(2):
        out.fill(0x5A)
        plan.run()
        gj.synchronize()
        assert np.array_equal(out.numpy(), orc.lookup_lower_bound(keys, probes))
    plan.close()
    idx.close()
