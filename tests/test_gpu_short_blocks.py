"""Block statistics in blocks of up to two samples per lane of a workgroup:
the lengths around both, blocks cut by the row's end, and negative zeros,
against the oracle bit for bit."""
import numpy as np
import pytest

import oracle as O
from mdsm_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [1, 2, 16, 255, 256, 257, 511, 512, 513, 1025])
@pytest.mark.parametrize("tail", [0, 1, 15])
def test_short_blocks_bitexact(L, tail):
    rows, nsamp = 3, 4 * L + min(tail, L - 1)
    rng = np.random.default_rng(L + tail)
    x = (rng.standard_normal((rows, nsamp)) * 3 + 7).astype(np.float32)
    x[0, : 2 * L] = -0.0
    d_x = abi.DeviceBuffer.from_numpy(x)
    nb = -(-nsamp // L)
    d_m, d_s = abi.DeviceBuffer(rows * nb * 8), abi.DeviceBuffer(rows * nb * 8)
    abi.block_stats(d_x.ptr, rows, nsamp, L, d_m.ptr, d_s.ptr)
    abi.synchronize()
    m, sd = O.block_stats(x, L)
    got_m, got_s = d_m.download(np.float64, (rows, nb)), d_s.download(np.float64, (rows, nb))
    assert np.array_equal(got_m, m) and np.array_equal(got_s, sd)
    assert not np.signbit(got_m[0, 0])  # sums start from +0
