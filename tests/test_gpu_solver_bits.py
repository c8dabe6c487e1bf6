"""The solver matrix from the free-column bits: rows that start at every place of
a 64-entry word, odd row counts (two rows a wavefront), rows of one chunk and of
seven, and boundary conditions changed in between; values, rows and columns must
equal the restriction of the equations matrix exactly, on the first pass (which
writes the columns) and on the next."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n", [(1, 1, 1), (2, 1, 3), (4, 3, 2)])
def test_restriction(gpu, n, precision):
    cm = gpu
    mesh = cm.RegularMesh.generate(2, n, jitter=0.1, seed=7)
    eq = cm.MooneyRivlinEquationsSet(mesh, 2.0, 6.0)
    eq.set_dofs(eq.undeformed_dofs() * 1.01)
    rng = np.random.default_rng(1)
    for count in (1, eq.n_rows // 3, eq.n_rows - 1):
        fixed = np.sort(rng.choice(eq.n_rows, count, replace=False))
        eq.set_boundary_conditions(fixed, np.zeros(count))
        free = np.ones(eq.n_rows, bool)
        free[fixed] = False
        number = np.cumsum(free) - 1
        for scale in (1.0, 1.02):
            eq.set_dofs(eq.undeformed_dofs() * scale)
            eq.residual_evaluate()
            eq.jacobian_evaluate(precision)
            eq.solver_matrices_assemble(precision)
            rp, ci = eq.matrix_structure()
            vals = eq.matrix_values_sp() if precision else eq.matrix_values()
            rows = np.repeat(np.arange(eq.n_rows), np.diff(rp))
            keep = free[rows] & free[ci]
            srp, sci = eq.solver_matrix_structure(0)
            got = eq.solver_matrix_values_sp() if precision else eq.solver_matrix_values()
            np.testing.assert_array_equal(got, vals[keep])
            np.testing.assert_array_equal(sci, number[ci[keep]])
            np.testing.assert_array_equal(np.diff(srp), np.bincount(number[rows[keep]], minlength=free.sum()))
    eq.destroy()
