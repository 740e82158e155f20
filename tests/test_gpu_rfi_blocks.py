"""The channel clipper on block lengths around its groups of blocks (64 blocks
of up to 256 samples, about 16384 samples of longer ones, one block past that),
and its rate where whole rows are flagged in a few long blocks."""
import numpy as np
import pytest

from mdsm_amd import abi

pytestmark = pytest.mark.gpu


def clip(d_x, ld, C, col0, n, d_fitted, cb, d_flags):
    abi.check(abi.lib().mdsm_rfi_channel_clip(d_x.ptr, ld, C, col0, n, d_fitted.ptr, cb, d_flags.ptr, None))


@pytest.mark.parametrize("cb", [1, 63, 256, 257, 1024, 8192, 16384, 16385, 40000])
@pytest.mark.parametrize("share", [0.1, 1.0])
def test_flagged_blocks_filled(cb, share):
    C, col0, n = 3, 5, 66 * min(cb, 1024) + 7 if cb < 8192 else 100003
    ld, nb = col0 + n + 9, -(-n // cb)
    rng = np.random.default_rng(cb)
    x = rng.standard_normal((C, ld)).astype(np.float32)
    fitted = rng.standard_normal(C)
    flags = (rng.random((C, nb)) < share).astype(np.uint8)
    flags[:, [0, nb - 1]] = [[1, 0], [0, 1], [1, 1]] if nb > 1 else [[1], [0], [1]]
    want = x.copy()
    toward_zero = np.where(np.abs(fitted.astype(np.float32).astype(np.float64)) > np.abs(fitted),
                           np.nextafter(fitted.astype(np.float32), np.float32(0)), fitted.astype(np.float32))
    for c in range(C):
        hit = np.repeat(flags[c] != 0, cb)[:n]
        want[c, col0:col0 + n][hit] = toward_zero[c]
    d_x = abi.DeviceBuffer.from_numpy(x)
    clip(d_x, ld, C, col0, n, abi.DeviceBuffer.from_numpy(fitted), cb, abi.DeviceBuffer.from_numpy(flags))
    abi.synchronize()
    assert np.array_equal(d_x.download(np.float32, x.shape), want)


def test_long_flagged_blocks_at_a_fill_s_rate():
    """One row of 2^24 samples in 64 flagged blocks: a plain fill of it by the
    whole card is the floor; 64 workgroups reach a fraction of its rate, a
    single wave some hundredth."""
    C, n, cb = 1, 1 << 24, 1 << 18
    d_x, d_f = abi.DeviceBuffer(n * 4), abi.DeviceBuffer.from_numpy(np.ones(C))
    d_g = abi.DeviceBuffer.from_numpy(np.ones((C, n // cb), np.uint8))

    def best(fn):
        times = []
        for _ in range(6):
            t = abi.Timer()
            t.start()
            for _ in range(5):
                fn()
            times.append(t.stop() / 5)
        return min(times[1:])

    fill = best(lambda: abi.check(abi.lib().mdsm_memset(d_x.ptr, 0, n * 4, None)))
    assert best(lambda: clip(d_x, n, C, 0, n, d_f, cb, d_g)) < 12 * fill
