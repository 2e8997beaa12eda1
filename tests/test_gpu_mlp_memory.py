"""Device memory of networks that only predict: weights in their forms and the
optimiser's state, not the buffer of partial gradients (21 MB at 34 inputs and 128
hidden units).  Gradients and training of such a handle work afterwards."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_prediction_keeps_no_gradient_buffer():
    from q_amd.mlp import MLP
    x = np.random.default_rng(0).normal(size=(100, 34)).astype(np.float32)
    t = np.full(100, 0.5, np.float32)
    MLP(34, 128, seed=0).forward(x)   # the device's scratch array exists from here on
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    nets = [MLP(34, 128, seed=k) for k in range(16)]
    for net in nets:
        net.forward(x)
    used = free - torch.cuda.mem_get_info()[0]
    print("MB a network", used / 16 / 2 ** 20)
    assert used < 16 * 8 * 2 ** 20
    loss, g = nets[0].grad(x, t)
    assert np.isfinite(loss) and np.abs(g).max() > 0
    assert nets[0].train(x, t, epochs=2, batch=50, lr=1e-3, seed=0) < 1.0
    for net in nets:
        net.close()
