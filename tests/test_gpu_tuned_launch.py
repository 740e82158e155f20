"""What the autotuners report can be had again by its number: a plan's on few
outputs (where the kernel without tiles, number 0, is the fastest by far) and
on many, and a batch's, which is no slower than the untuned batch."""
import numpy as np
import pytest

from mdsm_amd import abi

pytestmark = pytest.mark.gpu


def time_of(fn, inner=10):
    fn()
    times = []
    for _ in range(8):
        t = abi.Timer()
        t.start()
        for _ in range(inner):
            fn()
        times.append(t.stop() / inner)
    return min(times)


@pytest.mark.parametrize("C,M,N", [(256, 64, 8192), (256, 500, 60000)])
@pytest.mark.parametrize("dtype", [abi.F32, abi.U8])
def test_plan_number_launches_what_was_timed(dtype, C, M, N):
    s = abi.Survey.make(1500.0, -300.0 / C, C, 64e-6, 0.0, 0.1, M, N)
    p, q = abi.Plan(s, dtype), abi.Plan(s, dtype)
    d_x, d_y = abi.DeviceBuffer(C * p.min_ld * 4), abi.DeviceBuffer(M * N * 4)
    d_x.zero()
    v, ms = p.autotune(d_x.ptr, p.min_ld, d_y.ptr)
    assert p.variant == v
    q.set_variant(v)
    # (a launch timed alone carries 0.02 ms of events; pinned tiles take 0.13 ms)
    assert time_of(lambda: q.dedisperse(d_x.ptr, q.min_ld, d_y.ptr)) < 1.15 * ms + 0.01
    assert time_of(lambda: p.dedisperse(d_x.ptr, p.min_ld, d_y.ptr)) < 1.15 * ms + 0.01
    if M == 64:
        assert v == 0


# beams of few trials: 32-trial tiles, and pair sums of 40
@pytest.mark.parametrize("dtype,C,M,N", [(abi.F32, 512, 32, 300000), (abi.F16, 400, 30, 200000), (abi.U8, 256, 40, 150000)])
def test_batch_tuned_no_slower_than_untuned(dtype, C, M, N):
    beams = [abi.Survey.make(1500.0, -300.0 / C, C, 64e-6, 0.0, 0.02, M, N) for _ in range(2)]
    b, c = abi.Batch(beams, dtype), abi.Batch(beams, dtype)
    xs = [abi.DeviceBuffer(C * ld * 4) for ld in b.min_ld]
    ys = [abi.DeviceBuffer(M * N * 4) for _ in beams]
    for x in xs:
        x.zero()
    args = ([x.ptr for x in xs], list(b.min_ld), [y.ptr for y in ys])
    b.bind(*args)
    untuned = time_of(b.launch)
    v, _ = b.autotune(*args)
    c.set_variant(v)
    for tuned in (b, c):
        tuned.bind(*args)
        assert time_of(tuned.launch) < 1.05 * untuned
