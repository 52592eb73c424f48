"""Construction of the learned indexes on the GPU, at the edges of its kernels: placements of
less than one block's lines, of several blocks and of several steps per block; keys that
crowd at the end of the key range (lines past the last target) or leave long gaps; leaves
around the size from which a block instead of a wave fits them."""
import numpy as np
import pytest

from gpujoin_amd import _lib

pytestmark = pytest.mark.gpu


def _lookup_all(gj, keys, params, kind="learned_plr"):
    col = gj.DeviceArray.from_numpy(keys)
    idx = gj.Index(kind, col, host_column=keys, params=params)
    st = idx.stats()
    dp = col
    out = gj.DeviceArray(keys.size, np.uint32)
    idx.lookup(dp, out)
    gj.synchronize()
    got = out.numpy()
    idx.close()
    return got, st


def _targets(keys, line_keys):
    """floor((key - min) * mult / 2^64) in whole numbers, mult = floor(targets * 2^64 / (range + 1))."""
    targets = -(-keys.size // line_keys)
    span = int(keys[-1]) - int(keys[0])
    mult = min((targets << 64) // (span + 1), (1 << 64) - 1)
    mh, ml = np.uint64(mult >> 32), np.uint64(mult & 0xFFFFFFFF)
    off = (keys - keys[0]).astype(np.uint64)
    oh, ol = off >> np.uint64(32), off & np.uint64(0xFFFFFFFF)
    low = np.uint64(0xFFFFFFFF)
    mid = oh * ml + ((ol * ml) >> np.uint64(32))
    mid2 = ol * mh + (mid & low)
    return targets, (oh * mh + (mid >> np.uint64(32)) + (mid2 >> np.uint64(32))).astype(np.int64)


def _place(target, targets, n, cap):
    """The line of every key, one line after the other."""
    line = np.empty(n, np.int64)
    first = np.searchsorted(target, np.arange(targets + 1))
    pos, l = 0, 0
    while pos < n:
        end = min(int(first[min(l + 1, targets)]), pos + cap)
        line[pos:end] = l
        pos, l = end, l + 1
    return line, max(l, targets)


def _columns(kind, n, dtype, rng):
    top = (1 << 63) - 1 if dtype == np.uint64 else (1 << 32) - 2
    if kind == "uniform":
        k = rng.integers(0, top, n + n // 8 + 64)
    elif kind == "crowded_end":  # half of the keys in the last thousandth of the range
        k = np.concatenate([rng.integers(0, top, n // 2 + n // 8 + 64), top - rng.integers(1, top // 1000, n)])
    else:  # two far clusters: one gap of nearly all the lines
        k = np.concatenate([rng.integers(0, 8 * n, n), top - rng.integers(1, 8 * n, n)])
    k = np.unique(k.astype(np.uint64))
    pick = np.sort(rng.choice(k.size, n, replace=False))
    return k[pick].astype(dtype)


@pytest.mark.parametrize("dtype", [np.uint32, np.uint64])
@pytest.mark.parametrize("kind", ["uniform", "crowded_end", "gap"])
@pytest.mark.parametrize("n,line_keys", [(1, 10), (2, 1), (63, 10), (2047, 1), (2048, 1), (2049, 1), (70_001, 3),
                                         (300_007, 15)])
def test_placement(gj, gpu, dtype, kind, n, line_keys):
    keys = _columns(kind, n, dtype, np.random.default_rng(n + line_keys))
    got, st = _lookup_all(gj, keys, gj.index_params(learned_layout=_lib.LAYOUT_LINES, learned_line_keys=line_keys))
    assert np.array_equal(got, np.arange(n, dtype=np.uint32))
    if st["leaves"] == 0:  # root only: the placement can be restated
        targets, t = _targets(keys, line_keys)
        line, total = _place(t, targets, n, 15 if dtype == np.uint64 else 30)
        assert st["lines"] == total
        assert st["max_lines"] == int((line - t).max()) + 1
        assert abs(st["avg_lines"] - (1.0 + (line - t).mean())) < 1e-9


def test_placement_several_steps_per_block(gj, gpu):
    # more than 2048 blocks' worth of lines: every block scans its span in several steps
    n = (1 << 22) + 4099
    keys = _columns("uniform", n, np.uint64, np.random.default_rng(5))
    got, st = _lookup_all(gj, keys, gj.index_params(learned_layout=_lib.LAYOUT_LINES, learned_line_keys=1))
    assert np.array_equal(got, np.arange(n, dtype=np.uint32))
    targets, t = _targets(keys, 1)
    line, total = _place(t, targets, n, 15)
    assert st["leaves"] == 0 and st["lines"] == total and st["max_lines"] == int((line - t).max()) + 1


@pytest.mark.parametrize("kind", ["learned_plr", "learned_mlp"])
@pytest.mark.parametrize("dtype", [np.uint32, np.uint64])
@pytest.mark.parametrize("dist", ["uniform", "crowded_end", "gap"])
@pytest.mark.parametrize("n,leaf_bits,max_error", [(1, 1, 128), (4096, 1, 4096), (4097, 1, 128), (8300, 1, 4096),
                                                   (30_011, 2, 8), (30_011, 12, 2), (200_003, 3, 100_000)])
def test_leaves(gj, gpu, kind, dtype, dist, n, leaf_bits, max_error):
    keys = _columns(dist, n, dtype, np.random.default_rng(n + leaf_bits))
    got, st = _lookup_all(gj, keys, gj.index_params(learned_layout=_lib.LAYOUT_COLUMN, learned_leaf_bits=leaf_bits,
                                                    learned_max_error=max_error, mlp_steps=5), kind)
    assert np.array_equal(got, np.arange(n, dtype=np.uint32))
    assert st["leaves"] == 1 << leaf_bits
    assert st["max_window"] <= 2 * max_error + 2
    assert 0 <= st["fallback_keys"] <= n
    if max_error >= n:  # no leaf can be too wide
        assert st["fallback_keys"] == 0 and st["split_leaves"] == 0
