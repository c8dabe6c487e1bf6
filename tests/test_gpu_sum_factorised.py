"""Residual and Gauss-point records by one-dimensional sums: a block takes nine
elements, so the element counts end it at every fill (1, 8, 9, 10, 19 elements),
far from the origin too, where only differences from the element's centre keep
the derivatives' digits.  Bound: the oracle's own rounding there, the offset
over the element size times 2^-52 times the 27 terms of a sum."""
import numpy as np
import pytest

import oracle_lib as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0.0, 40.0])
@pytest.mark.parametrize("n", [(1, 1, 1), (2, 2, 2), (3, 3, 1), (5, 2, 1), (19, 1, 1)])
def test_residual_and_jacobian_against_the_oracle(gpu, n, offset):
    cm = gpu
    mesh = cm.RegularMesh.generate(2, n, jitter=0.1, seed=sum(n))
    mesh.coords = mesh.coords + offset
    eq = cm.MooneyRivlinEquationsSet(mesh, 2.0, 6.0)
    rng = np.random.default_rng(3)
    d = eq.undeformed_dofs()
    nu = 3 * mesh.n_nodes
    d[:nu] += 0.02 / max(n) * rng.uniform(-1, 1, nu)
    d[nu:] = 0.1 * rng.standard_normal(d.size - nu)
    eq.set_dofs(d)
    eq.residual_evaluate()
    eq.jacobian_evaluate(cm.OC_FP64)
    rp, ci = eq.matrix_structure()
    r = orc.mr_residual(mesh.elem_nodes, mesh.elem_nodes_l, mesh.coords, d, 2.0, 6.0)
    J = orc.mr_jacobian(mesh.elem_nodes, mesh.elem_nodes_l, mesh.coords, d, 2.0, 6.0, rp.astype(np.int64), ci)
    tol = 27 * 2.0 ** -52 * max(n) * (2.0 + offset) * 10
    assert np.linalg.norm(eq.residual() - r) <= tol * np.linalg.norm(r)
    assert np.linalg.norm(eq.matrix_values() - J) <= tol * np.linalg.norm(J)
    eq.destroy()
