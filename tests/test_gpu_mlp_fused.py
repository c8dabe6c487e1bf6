"""The fused network kernels at the edges of their tiles and limits (row tiles
of 32 and 128, column tiles of 32, outputs above and below eight, widths above
the fused limit), forward pass, loss and gradient against the float64 numpy
network with that test's tolerances."""
import numpy as np
import pytest

from test_gpu_mlp import numpy_grad, numpy_mlp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,layers,outputs,n", [
    (128, 4, 4, 1), (128, 4, 4, 33), (128, 4, 3, 4096), (32, 1, 8, 31), (33, 2, 9, 65), (30, 3, 40, 128),
    (127, 2, 128, 97), (5, 1, 1, 32), (130, 2, 4, 50), (16, 2, 4, 65536 + 129), (128, 4, 4, 65536 + 1)])
def test_network_matches_numpy(gpu, hidden, layers, outputs, n):
    from cm_amd.warm_start import FEATURE_SCALE, FEATURE_SHIFT, WarmStartMLP
    net = WarmStartMLP(hidden=hidden, layers=layers, outputs=outputs, seed=hidden + n)
    dims = [(9, hidden)] + [(hidden, hidden)] * (layers - 1) + [(hidden, outputs)]
    rng = np.random.default_rng(n)
    x = np.concatenate([rng.uniform(0, 1, (n, 3)), rng.uniform(-0.1, 0.1, (n, 3)), rng.uniform(0, 0.04, (n, 1)),
                        rng.uniform(1, 5, (n, 1)), rng.uniform(0, 10, (n, 1))], axis=1).astype(np.float32)
    t = rng.standard_normal((n, outputs)).astype(np.float32)
    p, shift, scale = net.parameters(), FEATURE_SHIFT.astype(np.float64), FEATURE_SCALE.astype(np.float64)
    y = net.forward(x)
    yref, _, _ = numpy_mlp(p, dims, x, shift, scale)
    assert np.abs(y - yref).max() / np.abs(yref).max() < 1e-5
    loss, g = net.gradient(x, t)
    lref, gref = numpy_grad(p, dims, x, t, shift, scale)
    assert abs(loss - lref) / lref < 1e-5
    assert np.linalg.norm(g - gref) / np.linalg.norm(gref) < 1e-4
    # smaller calls on the grown buffers
    assert np.array_equal(net.forward(x[:1]), net.forward(x[:1]))
    net.destroy()
