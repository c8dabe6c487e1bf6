"""Calls of shrinking and growing sizes on one network, whose staging buffers, device
copies and row tiles outlive a call: each against the float64 numpy network, with
the tolerances of test_gpu_mlp_fused, on inputs of its own."""
import numpy as np
import pytest

from test_gpu_mlp import numpy_grad, numpy_mlp

pytestmark = pytest.mark.gpu

# over and under 4 MiB of host arrays, two row tiles a block and one, its last rows
ROWS = [1, 120000, 33, 65537, 1, 5000, 31, 120001, 40]


def inputs(rng, n):
    return np.concatenate([rng.uniform(0, 1, (n, 3)), rng.uniform(-0.1, 0.1, (n, 3)), rng.uniform(0, 0.04, (n, 1)),
                           rng.uniform(1, 5, (n, 1)), rng.uniform(0, 10, (n, 1))], axis=1).astype(np.float32)


@pytest.mark.parametrize("hidden,layers,outputs", [(32, 2, 4), (40, 2, 12), (130, 1, 4)])
def test_sizes_in_turn(gpu, hidden, layers, outputs):
    from cm_amd.warm_start import FEATURE_SCALE, FEATURE_SHIFT, WarmStartMLP
    net = WarmStartMLP(hidden=hidden, layers=layers, outputs=outputs, seed=hidden)
    dims = [(9, hidden)] + [(hidden, hidden)] * (layers - 1) + [(hidden, outputs)]
    p, shift, scale = net.parameters(), FEATURE_SHIFT.astype(np.float64), FEATURE_SCALE.astype(np.float64)
    rng = np.random.default_rng(hidden)
    for n in ROWS:
        x = inputs(rng, n)
        yref, _, _ = numpy_mlp(p, dims, x, shift, scale)
        assert np.abs(net.forward(x) - yref).max() / np.abs(yref).max() < 1e-5, n
        x = inputs(rng, n)
        t = rng.standard_normal((n, outputs)).astype(np.float32)
        loss, g = net.gradient(x, t)
        lref, gref = numpy_grad(p, dims, x, t, shift, scale)
        assert abs(loss - lref) / lref < 1e-5, n
        assert np.linalg.norm(g - gref) / np.linalg.norm(gref) < 1e-4, n
    net.destroy()
