"""Blocks of dropped indexes are handed to the next build: indexes built, probed and dropped
by several threads on streams of their own, over columns whose blocks fit each other, must
each answer from their own structures, also when one is dropped right behind its lookup."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["btree", "learned_plr", "hash"])
def test_threads_share_blocks(gj, orc, gpu, kind):
    failures = []

    def work(t):
        try:
            stream = gj.Stream()
            for i in range(6):
                n = (1 << 21) + 7 * t + i  # 16 MiB and more: the lines layout
                keys = np.arange(n, dtype=np.uint64) * np.uint64(3 + t) + np.uint64(i)
                probes = keys[:: 5 + t].copy()
                probes[::7] += np.uint64(1)
                col, dp = gj.DeviceArray.from_numpy(keys), gj.DeviceArray.from_numpy(probes)
                out = gj.DeviceArray(probes.size, np.uint32)
                idx = gj.Index(kind, col, stream=stream)
                idx.lookup(dp, out, stream=stream)
                idx.close()  # waits for the lookup
                stream.synchronize()
                if not np.array_equal(out.numpy(), orc.lookup_lower_bound(keys, probes)):
                    failures.append((t, i))
        except Exception as e:  # noqa: BLE001
            failures.append((t, repr(e)))

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures


def test_sizes_that_the_pool_does_not_keep(gj, gpu):
    # a table beyond the pool's largest block, between two small indexes
    for n in (1, 1000, 1 << 24, 4096, 1):
        keys = np.arange(n, dtype=np.uint64) * np.uint64(5)
        col = gj.DeviceArray.from_numpy(keys)
        out = gj.DeviceArray(n, np.uint32)
        idx = gj.Index("hash", col)
        idx.lookup(col, out)
        gj.synchronize()
        assert np.array_equal(out.numpy(), np.arange(n, dtype=np.uint32))
        idx.close()
