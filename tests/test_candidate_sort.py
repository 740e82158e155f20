"""Candidate ordering by (dm_idx, sample): counts around the switch to digit
passes, key ranges of 0 to 64 bits, negative values, equal keys (whose payloads
all have to survive)."""
import numpy as np
import pytest

from mdsm_amd import abi


@pytest.mark.parametrize("n", [0, 1, 511, 512, 513, 20000])
@pytest.mark.parametrize("dm,sample", [((0, 1), (0, 1)), ((0, 1), (0, 1 << 22)), ((7, 600), (-5, 100000)),
                                       ((-2000, 2096), (0, 1 << 20)), ((-2000, 2097), (0, 1 << 20)),
                                       ((-(1 << 31), (1 << 31) - 1), (-(1 << 31), (1 << 31) - 1))])
def test_sorted_by_trial_and_sample(n, dm, sample):
    rng = np.random.default_rng(n)
    c = np.zeros(n, abi.CAND_DTYPE)
    c["dm_idx"] = rng.integers(*dm, n)
    c["sample"] = rng.integers(*sample, n)
    c["width_log2"] = np.arange(n)
    got = c.copy()
    abi.sort_candidates(got)
    want = c[np.lexsort((c["sample"], c["dm_idx"]))]
    assert np.array_equal(got["dm_idx"], want["dm_idx"]) and np.array_equal(got["sample"], want["sample"])
    assert np.array_equal(np.sort(got["width_log2"]), c["width_log2"])
    assert np.array_equal(c[got["width_log2"]], got)
