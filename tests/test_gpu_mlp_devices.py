"""Networks on two devices of one process: the training kernel's dynamic-LDS
limit belongs to a device, so a network of the second one has to set it too.
The gradients and the FP32 forward of both are the same bit for bit."""
import numpy as np
import pytest

from fsilbm3d_amd import _lib

pytestmark = pytest.mark.gpu


def test_a_network_on_a_second_device_trains():
    from fsilbm3d_amd.mlp import WarmStartNet
    lib = _lib.init()
    if lib.fsil_init(1) != 0:
        _lib.check(lib.fsil_init(0))
        pytest.skip("one device")
    rng = np.random.default_rng(3)
    X, Y = rng.standard_normal((200, 12)).astype(np.float32), rng.standard_normal((200, 3)).astype(np.float32)
    out = []
    try:
        for device in (0, 1):
            print(f"[gpu] network on device {device}", flush=True)
            _lib.check(lib.fsil_init(device))
            net = WarmStartNet(seed=7)
            loss, grad = net.loss_grad(X, Y)
            out.append((loss, grad, net.forward(X, bf16=False)))
            net.close()
    finally:
        _lib.check(lib.fsil_init(0))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
