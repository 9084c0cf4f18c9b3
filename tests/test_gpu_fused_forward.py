"""The one-kernel forward pass (surrogate.hip, mlp_forward_kernel): the layers' own products' bits at
the edges of its row blocks, its input paths (pinned, one copy, several pieces) and its widths.
PSIM_GEMM_CHOICE makes psim_mlp_forward run the products instead."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# row blocks of 32 and 64 with a remainder; 8192 / 8193: the rule between them on 256 CUs;
# 16384 / 16385: pinned / copied at 32 inputs; 32769: two pieces
@pytest.mark.parametrize("rows", [1, 31, 33, 64, 8192, 8193, 16384, 16385, 32769])
@pytest.mark.parametrize("n_in,hidden,layers", [(32, 512, 4), (7, 256, 1), (45, 256, 2)])
def test_fused_forward_gives_the_products_bits(monkeypatch, rows, n_in, hidden, layers):
    from psim_amd import surrogate
    net = surrogate.Surrogate(n_in=n_in, hidden=hidden, layers=layers, seed=3)
    x = np.random.default_rng(rows).uniform(-2, 2, size=(rows, n_in)).astype(np.float32)
    fused = net.predict(x)
    monkeypatch.setenv("PSIM_GEMM_CHOICE", "4")
    np.testing.assert_array_equal(fused, net.predict(x))
    net.close()


def test_fused_forward_reads_updated_weights_and_passes_infinities_on(monkeypatch):
    """The fragment-order weights follow a training step; infinite and NaN inputs come out as the
    products give them."""
    from psim_amd import surrogate
    net = surrogate.Surrogate(seed=8)
    rng = np.random.default_rng(1)
    x = rng.uniform(-1, 1, size=(300, surrogate.N_FEATURES)).astype(np.float32)
    before = net.predict(x)
    net.train_step(x, rng.uniform(-1, 1, size=300).astype(np.float32), 1e-2)
    x[3, 4], x[7, 0], x[9, 31] = np.inf, -np.inf, np.nan
    fused = net.predict(x)
    assert np.any(fused[10:] != before[10:])
    monkeypatch.setenv("PSIM_GEMM_CHOICE", "4")
    np.testing.assert_array_equal(fused, net.predict(x))
    net.close()
