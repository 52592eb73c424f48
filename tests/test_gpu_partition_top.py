"""Radix digits that reach past the key's top bit (ignore_bits is only held below the key's
width): the digit bits up there are zero, also where the first pass of two lies past the key
altogether, and every partition keeps the input order of its keys."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kb,ignore", [(8, 57), (8, 60), (8, 63), (4, 25), (4, 31)])
@pytest.mark.parametrize("bits,passes", [(8, 1), (8, 2), (10, 1), (10, 2), (14, 2)])
@pytest.mark.parametrize("m", [10007, 2_500_003])
def test_digits_past_the_key(gj, orc, gpu, kb, ignore, bits, passes, m):
    print(f"[case] kb={kb} ignore={ignore} bits={bits} passes={passes} m={m}", flush=True)
    rng = np.random.default_rng(ignore * 31 + bits)
    dt = np.uint64 if kb == 8 else np.uint32
    keys = rng.integers(0, np.iinfo(dt).max, size=m, dtype=dt)
    dropped = gj.DeviceArray.from_numpy(np.zeros(1, np.uint64))
    dk, dp, off, cnt = gj.partition(gj.DeviceArray.from_numpy(keys), m, bits, ignore, passes, dropped=dropped)
    gj.synchronize()
    assert int(dropped.numpy()[0]) == 0
    counts, ok, op = orc.partition(keys, bits, ignore)
    assert np.array_equal(cnt.numpy(), counts)
    starts = np.concatenate([[0], np.cumsum(counts)[:-1]]).astype(np.int64)
    idx = np.repeat(off.numpy().astype(np.int64) - starts, counts.astype(np.int64)) + np.arange(m, dtype=np.int64)
    assert np.array_equal(dk.numpy()[idx], ok)
    assert np.array_equal(dp.numpy()[idx], op)
