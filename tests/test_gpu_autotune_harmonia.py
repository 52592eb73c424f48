"""The index autotuner has one Harmonia candidate: the group widths no longer differ in kernel
or layout, so its choice does not hang on which of two equal timings came out shorter."""
import numpy as np
import pytest

from gpujoin_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kb,lanes", [(4, 8), (4, 32), (8, 16)])
def test_one_harmonia_candidate(gj, gpu, kb, lanes):
    print(f"[case] kb={kb} lanes={lanes}", flush=True)
    keys = gj.gen_build_keys(40000, kb, _lib.KEYS_UNIFORM, 0, 0x51 + kb)  # whole nodes of 32 keys
    col = gj.DeviceArray.from_numpy(keys)
    probes, _ = gj.gen_probes(keys, 20011, _lib.PROBES_UNIFORM, 1.0, 0.0, 0, 0x52)
    dp = gj.DeviceArray.from_numpy(probes)
    scratch = gj.DeviceArray(probes.size, np.uint32)
    picks = set()
    for _ in range(6):
        best, rate = gj.autotune_index("harmonia", col, dp, scratch, host_column=keys,
                                       base=gj.index_params(harmonia_group_lanes=lanes))
        assert rate > 0
        picks.add(best.harmonia_group_lanes)
    assert picks == {8}
