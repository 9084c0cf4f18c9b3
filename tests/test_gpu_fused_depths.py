"""The fused training kernels where LDS holds the activations of one row group only (surrogate.hip,
train_groups): the layers' own products' bits, which PSIM_GEMM_CHOICE makes the network run."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# hidden 256: two row groups up to 9 layers, one from 10 to the most a network has; 512: one from 5 to 9, none at
# 10 (layer by layer)
@pytest.mark.parametrize("rows", [1, 33, 1100])
@pytest.mark.parametrize("n_in,hidden,layers", [(20, 256, 10), (32, 256, 16), (32, 512, 5), (32, 512, 10)])
def test_deep_networks_give_the_products_bits(monkeypatch, rows, n_in, hidden, layers):
    from psim_amd import surrogate
    rng = np.random.default_rng(rows + layers)
    x = rng.uniform(-1, 1, size=(rows, n_in)).astype(np.float32)
    t = rng.uniform(-1, 1, size=rows).astype(np.float32)
    out = []
    for forced in (False, True):
        if forced:
            monkeypatch.setenv("PSIM_GEMM_CHOICE", "4")
        net = surrogate.Surrogate(n_in=n_in, hidden=hidden, layers=layers, seed=5)
        loss, grad = net.gradients(x, t)
        losses = [net.train_step(x, t, 1e-3) for _ in range(3)]  # eager, captured, replayed
        out.append((loss, grad, losses, net.params(), net.predict(x)))
        net.close()
    assert np.any(out[0][1] != 0)
    assert out[0][0] == out[1][0] and out[0][2] == out[1][2]
    for k in (1, 3, 4):
        np.testing.assert_array_equal(out[0][k], out[1][k])
