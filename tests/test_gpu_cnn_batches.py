"""The triage network's kernels take other splits of the work at large
batches: a batch of 128 full-size snippets gives the logits of its quarters
bit for bit (every snippet is summed on its own), and its gradients are the
mean of the quarters' (the BF16 roundings scale exactly by the batch ratio of
4; what is left is the order of FP32 sums of about 2^17 terms or fewer per
weight, 1e-5 of the norm)."""
import numpy as np
import pytest

import oracle
from mdsm_amd import abi

pytestmark = pytest.mark.gpu


def test_large_batch_equals_its_parts():
    H, W, B, parts = 64, 256, 128, 4
    rng = np.random.default_rng(77)
    x = abi.to_bf16_bits(rng.standard_normal((B, 2, H, W), dtype=np.float32))
    y = rng.integers(0, 2, B).astype(np.int32)
    p = np.zeros(oracle.cnn_param_count(H, W))
    fans = {"w1": 18, "w2": 144, "w3": 288, "fw1": 64 * 8 * 32, "fw2": 64}
    for name, a, b in oracle.cnn_param_slices(H, W):
        p[a:b] = rng.standard_normal(b - a) * (np.sqrt(2.0 / fans[name]) if name in fans else 0.05)

    def run(xs, ys):
        net = abi.TriageNet(H, W, len(xs))
        net.set_params(p)
        d_x, d_y = abi.DeviceBuffer.from_numpy(xs), abi.DeviceBuffer.from_numpy(ys)
        d_l, d_loss = abi.DeviceBuffer(len(xs) * 8), abi.DeviceBuffer(4)
        net.forward(d_x.ptr, len(xs), d_l.ptr)
        net.backward(d_y.ptr, len(xs), d_loss.ptr)
        g = net.grads()
        out = d_l.download(np.float32, (len(xs), 2)), g
        net.close()
        return out

    logits, grads = run(x, y)
    n = B // parts
    sub = [run(x[i * n:(i + 1) * n], y[i * n:(i + 1) * n]) for i in range(parts)]
    assert np.array_equal(logits, np.concatenate([s[0] for s in sub]))
    mean = np.mean([s[1].astype(np.float64) for s in sub], axis=0)
    for name, a, b in oracle.cnn_param_slices(H, W):
        err = np.linalg.norm(grads[a:b] - mean[a:b]) / np.linalg.norm(mean[a:b])
        assert err < 1e-5, (name, err)
