"""Shape numbers whose tiles are register windows now keep the surveys that
they took before: delay differences that fit DM tiles of 40 or 48 trials but
none of 64 or 32 (numbers 22 and 21), and a delay spread that fills LDS in
tiles of few samples only (number 12 of F32) -- plans and batches, against the
oracle bit for bit."""
import numpy as np
import pytest

import oracle as O
from mdsm_amd import abi

pytestmark = pytest.mark.gpu


def check(s, dtype, number):
    t, S = abi.delay_table(s)
    C, M, N = s.nchans, s.ndms, s.nsamp
    ld = -(-(N + S) // 4) * 4
    rng = np.random.default_rng(C)
    if dtype == abi.U8:
        x = rng.integers(0, 256, (C, ld)).astype(np.uint8)
        ref = O.dedisperse_u8(x, t, N)
    else:
        x = rng.standard_normal((C, ld)).astype(np.float32)
        if dtype != abi.F32:
            x = O.f32_to_f16(x)
        ref = (O.dedisperse_f16_pairs if dtype == abi.F16_PAIRS else O.dedisperse_f32seq)(x, t, N)
    assert abi.Plan(s, dtype).variant_channels(number) > 0
    assert np.array_equal(abi.dedisperse_host(s, x, dtype, number), ref)
    b = abi.Batch([s], dtype)
    b.set_variant(number)
    d_x, out = abi.DeviceBuffer.from_numpy(x), abi.DeviceBuffer(M * N * 4)
    for mode in (abi.BATCH_FLAT, abi.BATCH_PERSISTENT):
        b.set_mode(mode)
        b.dedisperse([d_x.ptr], [ld], [out.ptr])
        abi.synchronize()
        assert np.array_equal(out.download(np.float32, (M, N)), ref), mode


@pytest.mark.parametrize("C,M,step,number", [(64, 63, 0.15677701807, 22), (138, 78, 0.26534130849, 21)])
@pytest.mark.parametrize("dtype", [abi.U8, abi.F16_PAIRS])
def test_delay_differences_of_the_former_tiles(dtype, C, M, step, number):
    check(abi.Survey.make(1500.0, -300.0 / C, C, 64e-6, 0.0, step, M, 3000), dtype, number)


def test_delay_spread_of_the_former_tile():
    C, M, spread = 3, 2, 19900
    _, per_dm = abi.delay_table(abi.Survey.make(418.0, -20.0 / C, C, 51.2e-6, 0.0, 1000.0, M, 3000))
    s = abi.Survey.make(418.0, -20.0 / C, C, 51.2e-6, 0.0, 1000.0 * spread / per_dm, M, 3000)
    assert abs(abi.delay_table(s)[1] - spread) <= 1
    check(s, abi.F32, 12)
