"""Where psim_mlp_forward puts the results of networks that have no fused pass: the pinned buffer up to 2 MB
of them, a device buffer beyond.  psim_mlp_forward_noalloc, which has neither, gives the same bits."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

_F = ctypes.POINTER(ctypes.c_float)


def _noalloc(net, x):
    f = net._L.psim_mlp_forward_noalloc
    f.restype, f.argtypes = ctypes.c_int, [ctypes.c_void_p, _F, ctypes.c_int32, _F]
    y = np.full(x.shape[0], np.nan, np.float32)
    for r in range(0, x.shape[0], 20_000):
        piece = np.ascontiguousarray(x[r:r + 20_000])
        rc = f(net._h, piece.ctypes.data_as(_F), len(piece), y[r:].ctypes.data_as(_F))
        assert rc == 0, net._L.psim_mlp_last_error(net._h).decode()
    return y


# a width without a fused pass (the last sizes: 2 MB of results, one row more), and more inputs than the width
@pytest.mark.parametrize("n_in,hidden,rows", [(32, 128, 1), (32, 128, 300), (32, 128, 524_288), (32, 128, 524_289),
                                              (600, 512, 900)])
def test_results_of_layer_by_layer_passes(n_in, hidden, rows):
    from psim_amd import surrogate
    net = surrogate.Surrogate(n_in=n_in, hidden=hidden, layers=2, seed=4)
    x = np.random.default_rng(rows).uniform(-1, 1, size=(rows, n_in)).astype(np.float32)
    want = _noalloc(net, x)
    assert np.all(np.isfinite(want)) and np.any(want != 0)
    for _ in range(2):
        np.testing.assert_array_equal(net.predict(x), want)
    net.close()
