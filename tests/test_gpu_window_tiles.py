"""GPU parity of the register-window dedispersion tiles at their edges: time
tiles of 1280 samples, DM tiles of 32 trials (4 per wave), channel blocks of
6 (F32) and 8 (F16, U8), and delay slopes from several trials per window to
one (the reads end at 36 words), against the oracle bit for bit."""
import sys

import numpy as np
import pytest

import oracle as O
from mdsm_amd import abi

pytestmark = pytest.mark.gpu

# (nchans, ndms, nsamp, dmstep): about 0.1, 1.4, 4, 7, 16 and 60 samples per
# trial at the lowest channel of the 418 MHz band below
SHAPES = [(1, 1, 1, 0.1), (5, 3, 1279, 0.002), (6, 4, 1280, 0.03), (7, 5, 1281, 0.09), (8, 31, 2559, 0.15),
          (9, 32, 2561, 0.35), (17, 33, 700, 1.3), (16, 65, 4000, 0.09), (25, 37, 1300, 0.15)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype,variant", [(abi.F32, 12), (abi.F16, 12), (abi.U8, 2)])
def test_window_tiles_bitexact(shape, dtype, variant):
    C, M, N, step = shape
    s = abi.Survey.make(418.0, -20.0 / C, C, 51.2e-6, 0.0, step, M, N)
    t, S = abi.delay_table(s)
    print(f"[window tile] dtype {dtype} C={C} M={M} N={N} S={S}", flush=True, file=sys.stderr)
    rng = np.random.default_rng(C * 100 + M)
    ld = -(-(N + S) // 4) * 4
    if dtype == abi.U8:
        x = rng.integers(0, 256, (C, ld)).astype(np.uint8)
        ref = O.dedisperse_u8(x, t, N)
    else:
        x = (rng.standard_normal((C, ld)) * 3).astype(np.float32)
        if dtype == abi.F16:
            x = O.f32_to_f16(x)
        ref = O.dedisperse_f32seq(x, t, N) if dtype == abi.F32 else O.dedisperse_f16(x, t, N)
    assert np.array_equal(abi.dedisperse_host(s, x, dtype, variant), ref)
    b = abi.Batch([s, s], dtype)
    b.set_variant(variant)
    d_x = abi.DeviceBuffer.from_numpy(x)
    outs = [abi.DeviceBuffer(M * N * 4) for _ in range(2)]
    for mode in (abi.BATCH_FLAT, abi.BATCH_PERSISTENT):
        b.set_mode(mode)
        b.dedisperse([d_x.ptr] * 2, [ld] * 2, [o.ptr for o in outs])
        abi.synchronize()
        for o in outs:
            assert np.array_equal(o.download(np.float32, (M, N)), ref), mode
