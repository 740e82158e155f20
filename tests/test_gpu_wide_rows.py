"""GPU parity of the streaming passes that move four samples per access, at
the row lengths, offsets and strides where their whole groups end: channel
and block statistics, normalised storage, the median filter and the global
threshold, against the oracle bit for bit."""
import numpy as np
import pytest

import oracle as O
from mdsm_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ld,ldo,shift", [(1, 1, 1, 0), (3, 5, 4, 1), (4, 4, 7, 2), (1023, 1025, 1023, 3),
                                            (4096, 4096, 4096, 0), (4099, 4101, 4100, 1), (9001, 9001, 9002, 2)])
@pytest.mark.parametrize("name,dtype", [("f32", abi.F32), ("f16", abi.F16), ("u8", abi.U8)])
def test_normalise_rows(name, dtype, n, ld, ldo, shift):
    rng = np.random.default_rng(n + ld)
    C, size = 3, {"f32": 4, "f16": 2, "u8": 1}[name]
    raw = (rng.standard_normal((C, ld)) * 5 + 20).astype(np.float32)
    d_r = abi.DeviceBuffer.from_numpy(raw)
    d_m, d_s = abi.DeviceBuffer(C * 8), abi.DeviceBuffer(C * 8)
    abi.channel_stats(d_r.ptr, ld, C, n, d_m.ptr, d_s.ptr)
    m, sd = O.channel_stats(raw, n)
    assert np.array_equal(d_m.download(np.float64, (C,)), m) and np.array_equal(d_s.download(np.float64, (C,)), sd)
    np_dt = {"f32": np.float32, "f16": np.uint16, "u8": np.uint8}[name]
    off = shift * size if name != "f32" else 0  # output rows off the 4-byte grid
    d_o = abi.DeviceBuffer(off + C * ldo * size)
    d_o.zero()
    abi.normalise(d_r.ptr, ld, C, n, d_m.ptr, d_s.ptr, d_o.ptr + off, dtype, ldo)
    abi.synchronize()
    got = d_o.download(np_dt, (C, ldo), offset=off)
    ref = O.normalise(np.ascontiguousarray(raw[:, :n]), m, sd, name, n)
    assert np.array_equal(got[:, :n], np.asarray(ref).reshape(C, -1)[:, :n])
    assert not got[:, n:].any()


@pytest.mark.parametrize("nrows,nsamp", [(1, 1), (2, 2), (3, 5), (2, 6), (3, 7), (2, 1023), (3, 1025), (5, 4098)])
def test_median_and_threshold_rows(nrows, nsamp):
    rng = np.random.default_rng(nsamp)
    x = rng.standard_normal((nrows, nsamp)).astype(np.float32)
    x[:, ::3] = np.round(x[:, ::3])  # ties
    d_x, d_o = abi.DeviceBuffer.from_numpy(x), abi.DeviceBuffer(x.nbytes)
    abi.median_filter5(d_x.ptr, nrows, nsamp, d_o.ptr)
    assert np.array_equal(d_o.download(np.float32, x.shape), O.median_filter5(x))
    cap = nrows * nsamp
    d_c, d_n = abi.DeviceBuffer(cap * 16), abi.DeviceBuffer(4)
    abi.threshold_global(d_x.ptr, nrows, nsamp, 0.1, 0.9, 0.75, d_c.ptr, cap, d_n.ptr)
    c = abi.read_candidates(d_c, d_n, cap)
    od, ot, osnr, on = O.threshold_ref(x, 0.1, 0.9, 0.75)
    assert len(c) == on
    assert list(c["dm_idx"]) == list(od) and list(c["sample"]) == list(ot) and np.array_equal(c["snr"], osnr)


@pytest.mark.parametrize("nsamp,L", [(255, 100), (4096, 4096), (4097, 4096), (9000, 4095), (20001, 8191)])
def test_block_statistics(nsamp, L):
    x = (np.random.default_rng(L).standard_normal((3, nsamp)) * 4 + 1).astype(np.float32)
    nb = -(-nsamp // L)
    d_x, d_m, d_s = abi.DeviceBuffer.from_numpy(x), abi.DeviceBuffer(3 * nb * 8), abi.DeviceBuffer(3 * nb * 8)
    abi.block_stats(d_x.ptr, 3, nsamp, L, d_m.ptr, d_s.ptr)
    m, sd = O.block_stats(x, L)
    assert np.array_equal(d_m.download(np.float64, (3, nb)), m) and np.array_equal(d_s.download(np.float64, (3, nb)), sd)
