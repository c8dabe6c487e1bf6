"""The element-matrix pipelines at the element counts where a block's share
changes: one element, one short of the 256 compute units, one each, one over,
two each and one over, three each.  Batches of one-element meshes give every
count with elements of unit aspect."""
import numpy as np
import pytest

import oracle_lib as orc

pytestmark = pytest.mark.gpu


# tolerances of the Jacobian parity tests: FP64 1e-12, FP32 2e-6
@pytest.mark.parametrize("count", [1, 255, 256, 257, 513, 768])
@pytest.mark.parametrize("fp32", [False, True])
def test_jacobian(gpu, count, fp32):
    cm = gpu
    rng = np.random.default_rng(count)
    meshes = [cm.RegularMesh.generate(2, 1, jitter=0.1, seed=m) for m in range(count)]
    eq = cm.MooneyRivlinBatch(meshes, 2.0, 6.0)
    X = np.concatenate([m.coords for m in meshes], axis=1)
    lam = np.array([1.1, 1.1 ** -0.5, 1.1 ** -0.5])
    z = X * lam[:, None] + 0.01 * rng.uniform(-1, 1, X.shape)
    dofs = np.concatenate([z.ravel(), 0.5 * rng.standard_normal(8 * count)])
    eq.set_dofs(dofs)
    eq.jacobian_evaluate(cm.OC_FP32 if fp32 else cm.OC_FP64)
    rp, ci = eq.matrix_structure(0)
    J = eq.matrix_values_sp() if fp32 else eq.matrix_values()
    cq = np.concatenate([m.elem_nodes + 27 * k for k, m in enumerate(meshes)]).astype(np.int32)
    cl = np.concatenate([m.elem_nodes_l + 8 * k for k, m in enumerate(meshes)]).astype(np.int32)
    oJ = orc.mr_jacobian(cq, cl, X, dofs, 2.0, 6.0, rp.astype(np.int64), ci)
    assert np.linalg.norm(J - oJ) < (2e-6 if fp32 else 1e-12) * np.linalg.norm(oJ)
