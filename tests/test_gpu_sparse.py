"""Waves of which few lanes hold a probe to search for: the window search passes over the
rounds that serve none of them.  Only the lanes of one place in their quad, or one lane of
a wave, hold a key inside the column's range; the rest are outside it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["learned_plr", "learned_mlp", "radix_spline"])
@pytest.mark.parametrize("dt", [np.uint32, np.uint64])
@pytest.mark.parametrize("n", [17, 5003])
def test_few_live_lanes(gj, orc, gpu, kind, dt, n):
    rng = np.random.default_rng(n)
    keys = (np.cumsum(rng.integers(1, 30, n)) + 1000).astype(dt)
    col = gj.DeviceArray.from_numpy(keys)
    idx = gj.Index(kind, col, host_column=keys, params=gj.index_params(learned_layout=1, mlp_steps=5))
    m = 64 * 40
    lane = np.arange(m) % 64
    for live in [lane % 4 == r for r in range(4)] + [lane == v for v in (0, 17, 42, 63)] + [lane < 5]:
        probes = np.where(live, rng.choice(keys, m) + rng.integers(0, 2, m).astype(dt), dt(7)).astype(dt)
        want = orc.lookup_lower_bound(keys, probes)
        dp = gj.DeviceArray.from_numpy(probes)
        out = gj.DeviceArray(m, np.uint32)
        out.fill(0x5A)
        idx.lookup(dp, out)
        gj.synchronize()
        assert np.array_equal(out.numpy(), want)
    idx.close()
