"""The scratch that gj_partition asks for is what it uses: a histogram row for each of two
workgroups per CU, and nothing is written behind it."""
import ctypes as C

import numpy as np
import pytest

from gpujoin_amd import _lib

pytestmark = pytest.mark.gpu

GUARD = 4096


@pytest.mark.parametrize("kb,bits,passes", [(4, 10, 1), (8, 12, 1), (8, 11, 2), (4, 14, 2)])
# 65_530: two chunks for each XCD, fewer than the workgroups that pad
@pytest.mark.parametrize("m", [1, 4097, 65_530, 3_000_017])
def test_scratch_is_exact(gj, orc, gpu, kb, bits, passes, m):
    print(f"[case] kb={kb} bits={bits} passes={passes} m={m}", flush=True)
    p = _lib.PartitionParams(bits, 0, passes)
    need = _lib.call("gj_partition_scratch_bytes", m, kb, C.byref(p))
    if passes == 1:  # rows of two workgroups per CU, 256 CUs; the span sums and the starts
        assert need <= 2 * 256 * (4 << bits) + (8 << bits) + (1 << 14)
    dt = np.uint64 if kb == 8 else np.uint32
    keys = np.random.default_rng(bits + m).integers(0, np.iinfo(dt).max, size=m, dtype=dt)
    cap = _lib.call("gj_partition_capacity", m, kb, bits)
    dk, dp = gj.DeviceArray(cap, dt), gj.DeviceArray(cap, np.uint32)
    off, cnt = gj.DeviceArray(1 << bits, np.uint64), gj.DeviceArray(1 << bits, np.uint64)
    scratch = gj.DeviceArray.from_numpy(np.full(need + GUARD, 0xA5, np.uint8))
    col = gj.DeviceArray.from_numpy(keys)
    out = _lib.Partitioned(d_keys=dk.ptr, d_payloads=dp.ptr, d_offsets=off.ptr, d_counts=cnt.ptr, capacity=cap)
    _lib.check(_lib.call("gj_partition", col.ptr, m, kb, C.byref(p), C.byref(out), scratch.ptr, need, None))
    gj.synchronize()
    assert (scratch.numpy()[need:] == 0xA5).all()
    counts, ok, op = orc.partition(keys, bits, 0)
    assert np.array_equal(cnt.numpy(), counts)
    starts = np.concatenate([[0], np.cumsum(counts)[:-1]]).astype(np.int64)
    idx = np.repeat(off.numpy().astype(np.int64) - starts, counts.astype(np.int64)) + np.arange(m, dtype=np.int64)
    assert np.array_equal(dk.numpy()[idx], ok)
    assert np.array_equal(dp.numpy()[idx], op)
