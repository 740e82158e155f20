"""Untuned plans on rows shorter than a workgroup's 256 samples (from the four
samples of one lane on) and on few of its time blocks, against the oracle bit
for bit; and the same number of outputs in one time block and in eight, which
take the same time where all eight XCDs share the work."""
import numpy as np
import pytest

import oracle as O
from mdsm_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,M,N", [(5, 3, 1), (17, 9, 3), (3, 1, 4), (16, 5, 5), (33, 70, 7), (40, 300, 63),
                                   (31, 17, 255), (20, 131, 256), (9, 33, 513), (18, 30, 2305)])
@pytest.mark.parametrize("dtype", [abi.F32, abi.F16, abi.U8, abi.F16_PAIRS])
def test_short_rows_bitexact(dtype, C, M, N):
    s = abi.Survey.make(418.0, -20.0 / C, C, 51.2e-6, 1.0, 0.37, M, N)
    t, S = abi.delay_table(s)
    rng = np.random.default_rng(C + N)
    if dtype == abi.U8:
        x = rng.integers(0, 256, (C, N + S)).astype(np.uint8)
        ref = O.dedisperse_u8(x, t, N)
    else:
        x = (rng.standard_normal((C, N + S)) * 3).astype(np.float32)
        if dtype != abi.F32:
            x = O.f32_to_f16(x)
        ref = {abi.F32: O.dedisperse_f32seq, abi.F16: O.dedisperse_f16, abi.F16_PAIRS: O.dedisperse_f16_pairs}[dtype](x, t, N)
    assert np.array_equal(abi.dedisperse_host(s, x, dtype), ref)


@pytest.mark.parametrize("dtype", [abi.F32, abi.F16, abi.U8])
def test_few_time_blocks_use_every_xcd(dtype):
    def best(M, N):
        s = abi.Survey.make(1500.0, -300.0 / 256, 256, 64e-6, 0.0, 0.1, M, N)
        p = abi.Plan(s, dtype)
        d_x, d_y = abi.DeviceBuffer(256 * p.min_ld * 4), abi.DeviceBuffer(M * N * 4)
        d_x.zero()
        times = []
        for _ in range(6):
            t = abi.Timer()
            t.start()
            for _ in range(5):
                p.dedisperse(d_x.ptr, p.min_ld, d_y.ptr)
            times.append(t.stop() / 5)
        return min(times[1:])

    assert best(8000, 256) < 2 * best(1000, 2048)
