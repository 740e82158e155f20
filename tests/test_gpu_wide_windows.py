"""GPU parity of the 16-wave register windows, which surveys of whole rounds of
their tiles (64 trials x 1280 samples, 256 at a time) take: around a DM tile
and around channel blocks (12 of F32 and of pair sums, 16 of F16 and U8), as
plans and in both launch forms of a batch; and of the shape that an untuned
plan falls back to on a delay spread that no window holds, with more outputs
than the kernel without tiles takes.  Against the oracle bit for bit."""
import numpy as np
import pytest

import oracle as O
from mdsm_amd import abi

pytestmark = pytest.mark.gpu

TILES = 256 * 1280


def data(dtype, C, ld, t, N):
    rng = np.random.default_rng(C)
    if dtype == abi.U8:
        x = rng.integers(0, 256, (C, ld), np.uint8)
        return x, O.dedisperse_u8(x, t, N)
    x = rng.standard_normal((C, ld), np.float32)
    if dtype == abi.F32:
        return x, O.dedisperse_f32seq(x, t, N)
    x = O.f32_to_f16(x)
    return x, (O.dedisperse_f16_pairs if dtype == abi.F16_PAIRS else O.dedisperse_f16)(x, t, N)


# whole rounds of 200 or 256 tiles, at channel counts (around multiples of the
# block) where 64 trials per tile are the faster form
CASES = [(abi.F32, 12, 12, C, M, 200 * 1280 - 3) for C, M in ((36, 63), (37, 64), (47, 64))]
CASES += [(d, v, 16, C, M, N) for d, v in ((abi.F16, 12), (abi.U8, 2))
          for C, M, N in ((128, 63, TILES - 3), (129, 64, TILES), (143, 64, TILES - 1279), (128, 128, TILES - 5))]
CASES += [(d, 22, 12, C, M, N) for d in (abi.U8, abi.F16_PAIRS)
          for C, M, N in ((1, 63, TILES - 3), (11, 64, TILES), (12, 63, TILES - 1279), (13, 64, TILES - 1),
                          (24, 128, TILES - 3), (25, 127, TILES - 640))]


@pytest.mark.parametrize("dtype,number,block,C,M,N", CASES)
def test_wide_windows_bitexact(dtype, number, block, C, M, N):
    s = abi.Survey.make(1500.0, -300.0 / C, C, 64e-6, 0.0, 0.015, M, N)
    t, S = abi.delay_table(s)
    ld = -(-(N + S) // 4) * 4
    x, ref = data(dtype, C, ld, t, N)
    p = abi.Plan(s, dtype)
    assert p.variant_channels(number) == block
    p.set_variant(number)
    d_x = abi.DeviceBuffer.from_numpy(x)
    outs = [abi.DeviceBuffer(M * N * 4) for _ in range(2)]
    p.dedisperse(d_x.ptr, ld, outs[0].ptr)
    abi.synchronize()
    assert np.array_equal(outs[0].download(np.float32, (M, N)), ref)
    b = abi.Batch([s, s], dtype)
    b.set_variant(number)
    for mode in (abi.BATCH_FLAT, abi.BATCH_PERSISTENT):
        b.set_mode(mode)
        for o in outs:
            o.zero()
        b.dedisperse([d_x.ptr] * 2, [ld] * 2, [o.ptr for o in outs])
        abi.synchronize()
        for o in outs:
            assert np.array_equal(o.download(np.float32, (M, N)), ref), mode


@pytest.mark.parametrize("dtype", [abi.F32, abi.F16])
def test_untuned_fallback_shape_bitexact(dtype):
    C, M, N = 64, 100, 60000  # some 1000 samples of delay per trial
    s = abi.Survey.make(400.0, -2.0, C, 64e-6, 0.0, 2.2, M, N)
    p = abi.Plan(s, dtype)
    assert p.variant_channels(abi.preferred_variant(dtype)) == 0 and p.variant_channels(p.variant) > 0
    t, S = abi.delay_table(s)
    ld = -(-(N + S) // 4) * 4
    x, ref = data(dtype, C, ld, t, N)
    assert np.array_equal(abi.dedisperse_host(s, x, dtype), ref)
