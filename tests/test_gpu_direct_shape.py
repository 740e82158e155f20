"""Untuned plans with few outputs run the kernel without tiles: every storage
type against the oracle bit for bit, at channel counts around its groups of
16 (odd last channels of the pair sums among them), trials around its groups
of 4, and rows that end inside a lane's four samples."""
import numpy as np
import pytest

import oracle as O
from mdsm_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,M,N", [(1, 1, 256), (15, 3, 257), (16, 4, 258), (17, 5, 259), (33, 9, 1023), (64, 2, 5000)])
@pytest.mark.parametrize("dtype", [abi.F32, abi.F16, abi.U8, abi.F16_PAIRS])
def test_direct_shape_bitexact(dtype, C, M, N):
    s = abi.Survey.make(418.0, -20.0 / C, C, 51.2e-6, 1.0, 0.37, M, N)
    t, S = abi.delay_table(s)
    rng = np.random.default_rng(C + N)
    if dtype == abi.U8:
        x = rng.integers(0, 256, (C, N + S)).astype(np.uint8)
        ref = O.dedisperse_u8(x, t, N)
    else:
        x = (rng.standard_normal((C, N + S)) * 3).astype(np.float32)
        if dtype != abi.F32:
            x = O.f32_to_f16(x)
        ref = {abi.F32: O.dedisperse_f32seq, abi.F16: O.dedisperse_f16, abi.F16_PAIRS: O.dedisperse_f16_pairs}[dtype](x, t, N)
    assert np.array_equal(abi.dedisperse_host(s, x, dtype), ref)
