"""Delay spreads whose staged row takes all 160 KB of a CU's LDS (20480 words
twice for F32, 32768 and their bytes for U8): plans and both launch forms of a
batch against the oracle bit for bit."""
import numpy as np
import pytest

import oracle as O
from mdsm_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,number,spread", [(abi.F32, 12, 19160), (abi.U8, 2, 31448)])
def test_rows_of_all_lds(dtype, number, spread):
    C, M, N = 3, 2, 3000
    t, per_dm = abi.delay_table(abi.Survey.make(418.0, -20.0 / C, C, 51.2e-6, 0.0, 1000.0, M, N))
    s = abi.Survey.make(418.0, -20.0 / C, C, 51.2e-6, 0.0, 1000.0 * spread / per_dm, M, N)
    t, S = abi.delay_table(s)
    assert abs(S - spread) <= 1 and abi.Plan(s, dtype).variant_channels(number) == 1
    rng = np.random.default_rng(8)
    ld = -(-(N + S) // 4) * 4
    if dtype == abi.U8:
        x = rng.integers(0, 256, (C, ld)).astype(np.uint8)
        ref = O.dedisperse_u8(x, t, N)
    else:
        x = rng.standard_normal((C, ld)).astype(np.float32)
        ref = O.dedisperse_f32seq(x, t, N)
    d_x, out = abi.DeviceBuffer.from_numpy(x), abi.DeviceBuffer(M * N * 4)
    b = abi.Batch([s], dtype)
    for v in (0, number):
        assert np.array_equal(abi.dedisperse_host(s, x, dtype, v), ref), v
        b.set_variant(v)
        for mode in (abi.BATCH_FLAT, abi.BATCH_PERSISTENT):
            b.set_mode(mode)
            b.dedisperse([d_x.ptr], [ld], [out.ptr])
            abi.synchronize()
            assert np.array_equal(out.download(np.float32, (M, N)), ref), (v, mode)
