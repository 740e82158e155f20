"""Batches whose beams have few time tiles: every tile of every beam is
produced once however the groups and rotations spread them over the XCDs."""
import numpy as np
import pytest

import oracle as O
from mdsm_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles", [[1], [7, 8, 9], [41, 1, 17, 33], [2, 3, 5, 24, 25]])
@pytest.mark.parametrize("dtype", [abi.F32, abi.U8])
def test_batch_time_tiles(dtype, tiles):
    rng = np.random.default_rng(sum(tiles))
    beams, xs, refs = [], [], []
    for k, n in enumerate(tiles):
        C, M, N = 3 + k, 5 + 40 * k, 1280 * n - 3
        s = abi.Survey.make(418.0, -20.0 / C, C, 51.2e-6, 0.0, 0.05, M, N)
        t, S = abi.delay_table(s)
        L = -(-(N + S) // 4) * 4
        x = rng.integers(0, 256, (C, L)).astype(np.uint8) if dtype == abi.U8 else rng.standard_normal((C, L)).astype(np.float32)
        beams.append(s)
        xs.append(x)
        refs.append((O.dedisperse_u8 if dtype == abi.U8 else O.dedisperse_f32seq)(x, t, N))
    b = abi.Batch(beams, dtype)
    d_x = [abi.DeviceBuffer.from_numpy(x) for x in xs]
    outs = [abi.DeviceBuffer.from_numpy(np.full(r.shape, -1e30, np.float32)) for r in refs]
    for mode in (abi.BATCH_FLAT, abi.BATCH_PERSISTENT):
        b.set_mode(mode)
        b.dedisperse([d.ptr for d in d_x], [x.shape[1] for x in xs], [o.ptr for o in outs])
        abi.synchronize()
        for o, r in zip(outs, refs):
            assert np.array_equal(o.download(np.float32, r.shape), r), mode
