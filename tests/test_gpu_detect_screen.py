"""The boxcar detector's FP32 screen (thresholds from 4 on) keeps every FP64
candidate: large offsets against the noise, tiny and huge scales, infinities
and NaN, thresholds on both sides of the rule, rows that end inside a run --
candidates and S/N equal the oracle's."""
import numpy as np
import pytest

import oracle as O
from mdsm_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset,scale", [(0.0, 1.0), (1e6, 1.0), (-3e4, 0.01), (0.0, 1e-33), (1e30, 1e36), (5.0, 1e-6)])
@pytest.mark.parametrize("thresh,nsamp,special", [(3.9, 3000, False), (4.0, 3649, False), (4.5, 912, True),
                                                  (6.0, 7777, True)])
def test_screen_keeps_every_candidate(offset, scale, thresh, nsamp, special):
    rng = np.random.default_rng(int(nsamp + thresh * 10))
    L, rows = 1024, 4
    x = rng.standard_normal((rows, nsamp))
    for w in (1, 2, 5, 16, 64):
        for r in range(rows):
            t = rng.integers(0, nsamp - w)
            x[r, t:t + w] += thresh / np.sqrt(w) * rng.uniform(0.9, 1.6)
    x = (x * scale + offset).astype(np.float32)
    x[0, -3:] += np.float32(9 * scale)  # at the row's end
    nb = -(-nsamp // L)
    # the statistics of the clean rows; then single samples become special
    m, sd = O.block_stats(x, L)
    if special:
        x[1, 100], x[1, 500], x[2, 700], x[2, 701] = np.inf, -np.inf, np.nan, np.nan
    d_x = abi.DeviceBuffer.from_numpy(x)
    d_m, d_s = abi.DeviceBuffer.from_numpy(m), abi.DeviceBuffer.from_numpy(sd)
    cap = 1 << 16
    d_c, d_n = abi.DeviceBuffer(cap * 16), abi.DeviceBuffer(4)
    abi.detect(d_x.ptr, rows, nsamp, L, d_m.ptr, d_s.ptr, 7, thresh, d_c.ptr, cap, d_n.ptr)
    c = abi.read_candidates(d_c, d_n, cap)
    od, ot, ok, osnr, on = O.detect(x, L, 7, thresh, stats=(m, sd))
    assert len(c) == on
    assert np.array_equal(c["dm_idx"], od) and np.array_equal(c["sample"], ot)
    assert np.array_equal(c["width_log2"], ok) and np.array_equal(c["snr"], osnr)
