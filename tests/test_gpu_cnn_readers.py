"""Two threads reading one triage network: parameters and gradients, whose
values differ everywhere, come back whole from every one of 40 overlapping
reads (each read exchanges the layout on the device and downloads it)."""
import threading

import numpy as np
import pytest

from mdsm_amd import abi

pytestmark = pytest.mark.gpu


def test_parameters_and_gradients_read_by_two_threads():
    H, W, B = 32, 64, 4
    net = abi.TriageNet(H, W, B)
    net.init(5)
    rng = np.random.default_rng(6)
    d_x = abi.DeviceBuffer.from_numpy(abi.to_bf16_bits(rng.standard_normal((B, 2, H, W), dtype=np.float32)))
    d_y = abi.DeviceBuffer.from_numpy(rng.integers(0, 2, B).astype(np.int32))
    net.forward(d_x.ptr, B)
    net.backward(d_y.ptr, B)
    abi.synchronize()
    want = [net.params(), net.grads()]
    wrong = [0, 0]

    def read(k, get):
        for _ in range(40):
            wrong[k] += not np.array_equal(get(), want[k])

    threads = [threading.Thread(target=read, args=(k, g)) for k, g in enumerate((net.params, net.grads))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert wrong == [0, 0]
