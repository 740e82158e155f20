"""The global threshold where candidates are many: all of them, once each, at
row lengths around a thread's four samples and a wave's 256; a full list; and
one reservation per wave, whether it holds one candidate or one in two."""
import numpy as np
import pytest

from mdsm_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsamp", [1, 3, 255, 257, 1026, 5003])
@pytest.mark.parametrize("every", [1, 2, 7, 300])
def test_all_candidates_once(nsamp, every):
    rows, mean, rms, thresh = 3, 0.25, 1.5, 4.0
    rng = np.random.default_rng(nsamp + every)
    x = rng.standard_normal((rows, nsamp)).astype(np.float32)
    x.reshape(-1)[::every] += np.float32(50)
    r, t = np.nonzero(x.astype(np.float64) - mean >= rms * thresh)
    d_x, d_n = abi.DeviceBuffer.from_numpy(x), abi.DeviceBuffer(4)
    cap = rows * nsamp
    d_c = abi.DeviceBuffer(cap * 16)
    abi.threshold_global(d_x.ptr, rows, nsamp, mean, rms, thresh, d_c.ptr, cap, d_n.ptr)
    c = abi.read_candidates(d_c, d_n, cap)
    order = np.lexsort((c["sample"], c["dm_idx"]))
    assert np.array_equal(c["dm_idx"][order], r) and np.array_equal(c["sample"][order], t)
    assert np.array_equal(c["snr"][order], ((x[r, t].astype(np.float64) - mean) / rms).astype(np.float32))
    # a list with room for half: the count is the whole number, nothing is written past the room
    room = len(r) // 2
    mark = np.full(cap * 4, 0x5A5A5A5A, np.uint32)
    d_c.upload(mark)
    abi.threshold_global(d_x.ptr, rows, nsamp, mean, rms, thresh, d_c.ptr, room, d_n.ptr)
    abi.synchronize()
    assert d_n.download(np.uint32, (1,))[0] == len(r)
    assert np.array_equal(d_c.download(np.uint32, (cap * 4,))[room * 4:], mark[room * 4:])


def test_dense_candidates_cost_one_reservation_per_wave():
    rows, nsamp = 256, 1 << 15
    cap = rows * nsamp // 2
    d_c, d_n = abi.DeviceBuffer(cap * 16), abi.DeviceBuffer(4)

    def best(every):
        x = np.zeros((rows, nsamp), np.float32)
        x[:, ::every] = 50
        d_x = abi.DeviceBuffer.from_numpy(x)
        times = []
        for _ in range(6):
            t = abi.Timer()
            t.start()
            for _ in range(5):
                abi.threshold_global(d_x.ptr, rows, nsamp, 0.0, 1.0, 20.0, d_c.ptr, cap, d_n.ptr)
            times.append(t.stop() / 5)
        return min(times[1:])

    # a wave takes 256 samples: one candidate in each, or 128
    assert best(2) < 2 * best(256)
