"""More than 2^32 probes in one plain or hash-join lookup: a launch keeps to HIP's limit of
fewer than 2^32 threads, so the waves take further steps.  The probes repeat one block of 2^20, and so do the
row ids; the first and last blocks and those around 2^32 are looked at whole."""
import ctypes as C

import numpy as np
import pytest

from gpujoin_amd import _lib

pytestmark = pytest.mark.gpu

TILE = 1 << 20


@pytest.mark.parametrize("kind,approach", [("hash", "plain"), ("learned_plr", "plain"), ("binary_search", "plain"),
                                           ("btree", "plain"), ("no_op", "hj")])
def test_beyond_2_32_probes(gj, orc, gpu, kind, approach):
    print(f"[case] {kind} {approach}", flush=True)
    m = (1 << 32) + 300
    keys = np.arange(1, 5000, dtype=np.uint32) * np.uint32(7)
    tile = np.random.default_rng(3).choice(np.concatenate([keys, keys + np.uint32(1)]), TILE)
    want = orc.lookup_lower_bound(keys, tile)
    probes = gj.DeviceArray(m, np.uint32)
    _lib.check(_lib.call("gj_memcpy_htod", probes.ptr, tile.ctypes.data_as(C.c_void_p), tile.nbytes, None))
    done = TILE
    while done < m:
        n = min(done, m - done)
        _lib.check(_lib.call("gj_memcpy_dtod", probes.offset(done), probes.ptr, n * 4, None))
        done += n
    out = gj.DeviceArray(m, np.uint32)
    out.fill(0x5A)
    idx = gj.Index("btree" if kind == "no_op" else kind, gj.DeviceArray.from_numpy(keys))
    idx.lookup(probes, out, approach=approach)
    gj.synchronize()
    got = np.empty(TILE, np.uint32)
    for first in (0, TILE, m // 2 // TILE * TILE, (1 << 32) - TILE, 1 << 32):
        n = min(TILE, m - first)
        _lib.check(_lib.call("gj_memcpy_dtoh", got.ctypes.data_as(C.c_void_p), out.offset(first), n * 4, None))
        assert np.array_equal(got[:n], want[:n]), first
    idx.close()
    probes.free()
    out.free()
