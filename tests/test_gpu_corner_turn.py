"""GPU parity of the register corner turn at its edges: spectra counts around
its 256-spectra blocks and 4-sample groups, channel counts of 8 and 16 and
not, beams that split a channel group, packed data off the access size."""
import numpy as np
import pytest

import oracle as O
from mdsm_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nspec", [1, 3, 4, 255, 257, 2051])
@pytest.mark.parametrize("nchans,nbeams,skew", [(8, 1, 0), (16, 1, 0), (12, 2, 0), (20, 2, 0), (64, 3, 0), (16, 1, 4)])
@pytest.mark.parametrize("nbits", [1, 2, 4, 8, 16, 32])
def test_unpack_corner_turn_edges(nbits, nchans, nbeams, skew, nspec):
    ctot, col0 = nchans * nbeams, 3
    rng = np.random.default_rng(nbits * 1000 + ctot + nspec)
    raw = rng.integers(0, 256, ctot * nbits // 8 * nspec).astype(np.uint8)
    if nbits == 32:
        raw = rng.standard_normal(ctot * nspec).astype(np.float32).view(np.uint8)
    ld = col0 + nspec + 2
    d_p = abi.DeviceBuffer(raw.nbytes + skew)
    d_p.upload(raw, skew)
    d_o = abi.DeviceBuffer(nbeams * nchans * ld * 4)
    d_o.zero()
    abi.unpack_corner_turn(d_p.ptr + skew, nbits, nspec, nchans, nbeams, d_o.ptr, ld, None, col0)
    abi.synchronize()
    got = d_o.download(np.float32, (nbeams, nchans, ld))
    v = O.sigproc_unpack(raw.tobytes(), nbits, ctot * nspec).reshape(nspec, nbeams, nchans)
    ref = np.zeros_like(got)
    ref[:, :, col0:col0 + nspec] = np.transpose(v, (1, 2, 0))
    assert np.array_equal(got, ref)
