"""The fused training kernels (surrogate.hip: mlp_train_kernel, mlp_grad_kernel, adam_fused_kernel): the
layers' own products' bits, which PSIM_GEMM_CHOICE makes the network run, at the edges of their row
blocks, chunks and splits, and for widths and depths at the ends of what they take."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# one row; chunks of 32 rows with a remainder; 4096 / 4097: 16 or 32 rows a block on 256 CUs, ragged
# splits; 16385: inputs copied instead of read from pinned memory
@pytest.mark.parametrize("rows", [1, 16, 33, 1024, 1100, 4096, 4097, 8200, 16385])
@pytest.mark.parametrize("n_in,hidden,layers", [(32, 512, 4), (32, 512, 1), (20, 256, 9), (7, 512, 9)])
def test_fused_gradients_and_steps_give_the_products_bits(monkeypatch, rows, n_in, hidden, layers):
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
        out.append((loss, grad, losses, net.params(), net.predict(x[:40])))
        net.close()
    assert out[0][0] == out[1][0] and out[0][2] == out[1][2]
    for k in (1, 3, 4):
        np.testing.assert_array_equal(out[0][k], out[1][k])
