"""RadixSpline over keys that crowd under few prefixes of its radix table, where a sample of the
knots replaces the table: fewer knots than samples, several per sample and a partial last
group, probes on, next to and far from keys."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.uint32, np.uint64])
@pytest.mark.parametrize("n", [2, 3, 33, 5000, 90_001, 400_009])
@pytest.mark.parametrize("max_error", [1, 32])
@pytest.mark.parametrize("bits", [1, 6, 18])
def test_crowded_prefixes(gj, orc, gpu, dt, n, max_error, bits):
    rng = np.random.default_rng(n + bits)
    top = np.iinfo(dt).max
    steps = np.where(rng.random(n) < 0.5, rng.integers(1, 3, n), rng.integers(1, 4000, n))
    keys = (np.uint64(5) + np.cumsum(steps).astype(np.uint64)).astype(dt)  # uneven, and low in the range
    keys[-1] = top - dt(1)  # one far key: all others share the first prefixes
    assert (np.diff(keys.astype(np.float64)) > 0).all()
    near = rng.choice(keys, 3000)
    probes = rng.permutation(np.concatenate([near, near + dt(1), near - dt(1), rng.integers(0, top, 500, dtype=dt),
                                             np.array([0, 1, top, top - 1, top - 2], dtype=dt)]))
    col, dp = gj.DeviceArray.from_numpy(keys), gj.DeviceArray.from_numpy(probes)
    out = gj.DeviceArray(probes.size, np.uint32)
    idx = gj.Index("radix_spline", col, params=gj.index_params(rs_radix_bits=bits, rs_max_error=max_error, rs_lds_bits=1))
    want = orc.lookup_lower_bound(keys, probes)
    for approach in ("plain", "bws", "partitioning"):
        out.fill(0x5A)
        idx.lookup(dp, out, approach=approach)
        gj.synchronize()
        assert np.array_equal(out.numpy(), want), approach
    idx.close()
