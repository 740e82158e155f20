"""GPU parity of the register windows over pair sums (time tiles of 1280
samples, DM tiles of 64 trials, blocks of 12 channels) and of the eight-wave
forms that surveys of few trials or wide delay spreads take, against the
oracle bit for bit."""
import numpy as np
import pytest

import oracle as O
from mdsm_amd import abi

pytestmark = pytest.mark.gpu


def reference(dtype, C, L, t, N, seed):
    rng = np.random.default_rng(seed)
    if dtype == abi.U8:
        x = rng.integers(0, 256, (C, L)).astype(np.uint8)
        return x, O.dedisperse_u8(x, t, N)
    x = (rng.standard_normal((C, L)) * 3).astype(np.float32)
    if dtype == abi.F32:
        return x, O.dedisperse_f32seq(x, t, N)
    x = O.f32_to_f16(x)
    return x, (O.dedisperse_f16_pairs if dtype == abi.F16_PAIRS else O.dedisperse_f16)(x, t, N)


# (nchans, ndms, nsamp, dmstep) on 1500 - 300 MHz: one block, its remainders,
# an odd last channel, several DM tiles, delay slopes that reopen windows
@pytest.mark.parametrize("C,M,N,step", [(1, 1, 1, 0.1), (2, 3, 1279, 0.05), (11, 63, 1280, 0.02), (12, 64, 1281, 0.018),
                                        (13, 65, 2561, 0.018), (37, 130, 700, 0.05), (256, 100, 3001, 0.4)])
@pytest.mark.parametrize("dtype", [abi.U8, abi.F16_PAIRS])
def test_window_pairs_bitexact(dtype, C, M, N, step):
    s = abi.Survey.make(1500.0, -300.0 / C, C, 64e-6, 0.0, step, M, N)
    t, S = abi.delay_table(s)
    ld = -(-(N + S) // 4) * 4
    x, ref = reference(dtype, C, ld, t, N, C * 100 + M)
    assert abi.Plan(s, dtype).variant_channels(22) > 0
    assert np.array_equal(abi.dedisperse_host(s, x, dtype, 22), ref)
    b = abi.Batch([s, s], dtype)
    b.set_variant(22)
    d_x = abi.DeviceBuffer.from_numpy(x)
    outs = [abi.DeviceBuffer(M * N * 4) for _ in range(2)]
    for mode in (abi.BATCH_FLAT, abi.BATCH_PERSISTENT):
        b.set_mode(mode)
        b.dedisperse([d_x.ptr] * 2, [ld] * 2, [o.ptr for o in outs])
        abi.synchronize()
        for o in outs:
            assert np.array_equal(o.download(np.float32, (M, N)), ref), mode


# untuned: 20 and 90 trials of just over 256 tiles of 64 trials; and a shape set by number
# whose 64 trials spread over more samples than an LDS row holds
@pytest.mark.parametrize("C,M,N,step,number", [(13, 20, 330001, 0.05, False), (7, 90, 170001, 0.002, False),
                                               (5, 64, 1300, 9.0, True)])
@pytest.mark.parametrize("dtype", [abi.F32, abi.F16, abi.U8, abi.F16_PAIRS])
def test_eight_wave_forms_bitexact(dtype, C, M, N, step, number):
    if number and dtype == abi.F16_PAIRS:
        pytest.skip("the pair sums have no such row: few delay differences per pair")
    s = abi.Survey.make(418.0, -20.0 / C, C, 51.2e-6, 0.0, step, M, N)
    t, S = abi.delay_table(s)
    ld = -(-(N + S) // 4) * 4
    x, ref = reference(dtype, C, ld, t, N, C)
    variant = (2 if dtype == abi.U8 else 12) if number else 0
    assert np.array_equal(abi.dedisperse_host(s, x, dtype, variant), ref)
    b = abi.Batch([s], dtype)
    b.set_variant(variant)
    d_x, out = abi.DeviceBuffer.from_numpy(x), abi.DeviceBuffer(M * N * 4)
    for mode in (abi.BATCH_FLAT, abi.BATCH_PERSISTENT):
        b.set_mode(mode)
        b.dedisperse([d_x.ptr], [ld], [out.ptr])
        abi.synchronize()
        assert np.array_equal(out.download(np.float32, (M, N)), ref), mode
