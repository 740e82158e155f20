"""Untuned plans on few channels, where a register-window tile's workgroups
wait for their stores longer than the adds win: the untuned launch takes no
more than 1.06 times as long as the shape set by number that overlaps both
(1.08 to 1.2 times where the choice weighed the adds alone)."""
import numpy as np
import pytest

from mdsm_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,C,M,N,step,number", [(abi.F16_PAIRS, 64, 4000, 50000, 0.01, 20),
                                                     (abi.U8, 64, 4000, 50000, 0.01, 21),
                                                     (abi.F16, 16, 200, 20000, 0.1, 15)])
def test_untuned_near_the_better_shape(dtype, C, M, N, step, number):
    s = abi.Survey.make(418.0, -20.0 / C, C, 51.2e-6, 0.0, step, M, N)
    p = abi.Plan(s, dtype)
    assert p.variant_channels(number) > 0
    d_x, d_y = abi.DeviceBuffer(C * p.min_ld * 2), abi.DeviceBuffer(M * N * 4)
    d_x.zero()

    def best(v):
        p.set_variant(v)
        times = []
        for _ in range(8):
            t = abi.Timer()
            t.start()
            for _ in range(8):
                p.dedisperse(d_x.ptr, p.min_ld, d_y.ptr)
            times.append(t.stop() / 8)
        return min(times[1:])

    assert best(0) < 1.06 * best(number)
