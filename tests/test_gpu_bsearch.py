"""Binary search by lines: columns of a bucket of 8 and 9 keys (where lines take over), of a
partial last line, with runs of equal keys across lines and buckets (the first of them is
the answer), with keys that crowd at one end of their bucket, and probes in both orders."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _column(kind, n, dt, rng):
    top = np.iinfo(dt).max
    if kind == "spread":
        k = rng.integers(0, top, n, dtype=dt, endpoint=True)
    elif kind == "runs":  # runs of 1 to 300 equal keys
        k = np.repeat(rng.integers(0, top, n, dtype=dt), rng.integers(1, 300, n))[:n]
    elif kind == "equal":
        k = np.full(n, 7, dtype=dt)
    else:  # powers: nearly all keys of a bucket close to its start
        k = (float(top) * rng.random(n) ** 40).astype(dt)
    return np.sort(k)


@pytest.mark.parametrize("dt", [np.uint32, np.uint64])
@pytest.mark.parametrize("kind", ["spread", "runs", "equal", "crowded"])
@pytest.mark.parametrize("n", [1, 5, 1000, 8192, 8193, 9217, 16384, 16385, 18433, 40_009, 131_072, 300_007])
def test_first_of_equal_keys(gj, orc, gpu, dt, kind, n):
    rng = np.random.default_rng(n)
    keys = _column(kind, n, dt, rng)
    top = np.iinfo(dt).max
    near = rng.choice(keys, 5000)
    probes = np.concatenate([near, near + dt(1), near - dt(1), rng.integers(0, top, 999, dtype=dt, endpoint=True),
                             np.array([0, 1, top, top - 1, keys[0], keys[-1]], dtype=dt)])
    col = gj.DeviceArray.from_numpy(keys)
    idx = gj.Index("binary_search", col)
    for order in ("shuffled", "sorted"):
        p = rng.permutation(probes) if order == "shuffled" else np.sort(probes)
        want = orc.lookup_lower_bound(keys, p)
        assert (want[np.isin(p, keys)] == np.searchsorted(keys, p[np.isin(p, keys)])).all()
        dp = gj.DeviceArray.from_numpy(p)
        out = gj.DeviceArray(p.size, np.uint32)
        for approach in ("plain", "bws", "partitioning"):
            out.fill(0x5A)
            idx.lookup(dp, out, approach=approach)
            gj.synchronize()
            assert np.array_equal(out.numpy(), want), (approach, order)
    idx.close()
