"""The MLP's kernels at the edges of their tiles (16 rows, 16 units, 64 and
128 inputs) and on both sides of the fused network's limits (128 inputs, 128
hidden units), against the same network in 64 bits.

Tolerances: a product of at most 129 FP32 terms is off by at most 129 x 2^-24
= 8e-6 of its terms' magnitudes and sigmoid's slope is 1/4, so outputs are
held to 2e-5; a gradient block is a sum of such terms, held to 1e-4 of its
largest element."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (3, 16, 15), (34, 128, 16), (64, 127, 17), (65, 100, 257), (128, 17, 4097), (129, 128, 33),
          (8, 129, 300)]


def network(n_in, hidden, rows):
    from q_amd.mlp import MLP
    rng = np.random.default_rng(n_in * 1000 + hidden)
    m = MLP(n_in, hidden, seed=5)
    p = m.params
    p += rng.normal(0, 0.05, p.size).astype(np.float32)   # biases are zero at first
    m.params = p
    x = rng.normal(size=(rows, n_in)).astype(np.float32)
    t = rng.uniform(size=rows).astype(np.float32)
    return m, x, t


def reference(m, x, t):
    ws = [torch.tensor(np.array(a)) for a in m.split()]
    ws = [w.to(torch.bfloat16) if k % 2 == 0 else w for k, w in enumerate(ws)]
    ws = [w.double().requires_grad_(True) for w in ws]
    h = torch.nn.functional.silu(torch.tensor(x).double() @ ws[0].T + ws[1])
    h = torch.nn.functional.silu(h @ ws[2].T + ws[3])
    y = torch.sigmoid(h @ ws[4].T + ws[5])[:, 0]
    loss = ((y - torch.tensor(t).double()) ** 2).mean()
    loss.backward()
    return y.detach().numpy(), float(loss), [w.grad.numpy() for w in ws]


@pytest.mark.parametrize("n_in,hidden,rows", SHAPES)
def test_shapes(n_in, hidden, rows):
    m, x, t = network(n_in, hidden, rows)
    y, loss, grads = reference(m, x, t)
    assert np.abs(m.forward(x) - y).max() < 2e-5
    l, g = m.grad(x, t)
    assert abs(l - loss) < 2e-5
    for a, b in zip(m.split(g), grads):
        assert np.abs(a - b).max() <= 1e-4 * np.abs(b).max() + 1e-12
    # one minibatch of all rows, in a shuffled order: the first Adam step moves
    # a parameter by lr g / (|g| + eps) (gradients near rounding left out)
    p0, lr = m.params, 1e-3
    assert abs(m.train(x, t, epochs=1, batch=rows, lr=lr, seed=3) - loss) < 2e-5
    big = np.abs(g) > 1e-3 * np.abs(g).max()
    step = lr * g / (np.abs(g) + 1e-8)
    assert np.abs((p0 - m.params) - step)[big].max() < 2e-5 * lr + 2.0 ** -23 * np.abs(p0).max()
    m.close()
