"""Meshes whose first and last nodes belong to no element, as the C boundary
takes them: their rows are empty and stand at both ends of the matrix.  The
answers must be those of the elements, and the unused DOFs stay as they were,
fixed or free."""
import numpy as np
import pytest

import oracle_lib as orc
from cm_amd.mesh import RegularMesh, UserMesh

pytestmark = pytest.mark.gpu


def with_unused_nodes(order, n, seed):
    """A jittered mesh with one more node before and after the others, of each component."""
    m = RegularMesh.generate(order, n, jitter=0.1, seed=seed)
    xyz = np.pad(m.coords, ((0, 0), (1, 1)), constant_values=7.0)
    u = UserMesh(order, (m.elem_nodes + 1).astype(np.int32), np.ascontiguousarray(xyz), np.arange(m.n_nodes + 2))
    if order == 2:
        u.elem_nodes_l = (m.elem_nodes_l + 1).astype(np.int32)
        u.node_user_numbers_l = np.arange(m.n_nodes_l + 2)
    return m, u


@pytest.mark.parametrize("fix_unused", [False, True])
@pytest.mark.parametrize("n", [(1, 1, 1), (3, 2, 2)])
def test_newton(gpu, n, fix_unused):
    cm = gpu
    m, u = with_unused_nodes(2, n, 5)
    nq = u.n_nodes
    eq = cm.MooneyRivlinEquationsSet(u, 2.0, 6.0)
    unused = np.array([0, nq - 1, nq, 2 * nq - 1, 2 * nq, 3 * nq - 1, 3 * nq, eq.n_rows - 1])
    faces = [m.face_nodes(0, 0) + 1, nq + m.face_nodes(1, 0) + 1, 2 * nq + m.face_nodes(2, 0) + 1,
             m.face_nodes(0, 1) + 1]
    values = np.concatenate([np.zeros(sum(len(f) for f in faces[:3])), np.full(len(faces[3]), 1.05)])
    fixed = np.concatenate(faces)
    d = eq.undeformed_dofs()
    d[unused] = np.arange(1, 9)
    eq.set_dofs(d)
    for precision in (cm.OC_FP64, cm.OC_FP32):  # every shape of the matrix products
        eq.autotune(precision)
    if fix_unused:
        fixed, values = np.concatenate([fixed, unused]), np.concatenate([values, d[unused]])
    eq.set_boundary_conditions(fixed, values)
    eq.load_increment_apply(1, 1)
    ref = eq.residual_norm()
    for precision in (cm.OC_FP32, cm.OC_FP64):
        start = eq.get_dofs()
        st = eq.newton_solve(cm.newton_options(solution_tolerance=0.0, relative_tolerance=0.0,
                                               absolute_tolerance=1e-10 * ref, krylov_restart=200,
                                               krylov_relative_tolerance=1e-4, jacobian_precision=precision,
                                               preconditioner=cm.OC_PRECONDITIONER_BLOCK_TRIANGULAR,
                                               maximum_iterations=12))
        assert st["converged"], st
        got = eq.get_dofs()
        r = orc.mr_residual(u.elem_nodes, u.elem_nodes_l, u.coords, got, 2.0, 6.0)
        r[fixed] = 0.0
        assert np.linalg.norm(r) <= 1.05e-10 * ref
        assert np.array_equal(got[unused], d[unused])
        eq.set_dofs(start)
    eq.destroy()


def check_restriction(eq, fixed, precision):
    """The solver matrix equals the equations matrix without the fixed rows and columns."""
    eq.solver_matrices_assemble(precision)
    rp, ci = eq.matrix_structure()
    vals = eq.matrix_values_sp() if precision else eq.matrix_values()
    free = np.ones(eq.n_rows, bool)
    free[fixed] = False
    rows = np.repeat(np.arange(eq.n_rows), np.diff(rp))
    keep = free[rows] & free[ci]
    number = np.cumsum(free) - 1
    srp, sci = eq.solver_matrix_structure(0)
    assert np.array_equal(eq.solver_matrix_values_sp() if precision else eq.solver_matrix_values(), vals[keep])
    assert np.array_equal(sci, number[ci[keep]])
    assert np.array_equal(np.diff(srp), np.bincount(number[rows[keep]], minlength=free.sum()))


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n", [(1, 1, 1), (2, 3, 1)])
def test_solver_matrix(gpu, n, precision):
    """With the last rows free and empty, and without them; odd and even row counts."""
    cm = gpu
    _, u = with_unused_nodes(2, n, 7)
    eq = cm.MooneyRivlinEquationsSet(u, 2.0, 6.0)
    eq.set_dofs(eq.undeformed_dofs() * 1.01)
    eq.residual_evaluate()
    eq.jacobian_evaluate(precision)
    for fixed in ([], [1], [0, 2, eq.n_rows - 1]):
        eq.set_boundary_conditions(fixed, np.zeros(len(fixed)))
        for _ in range(2):  # with the columns, then the values alone
            check_restriction(eq, fixed, precision)
    eq.destroy()


@pytest.mark.parametrize("n", [(2, 2, 2), (5, 4, 3)])
def test_laplace(gpu, n):
    """Assembly, solver matrix and solve (bound as in test_gpu_arnoldi)."""
    cm = gpu
    m, u = with_unused_nodes(1, n, 3)
    field = np.array([0.3, -0.7, 0.2]) @ u.coords + 0.1
    boundary = 1 + np.unique(np.concatenate([m.face_nodes(a, side) for a in range(3) for side in (0, 1)]))
    eq = cm.LaplaceEquationsSet(u)
    eq.assemble()
    rp, ci = orc.pattern([(u.n_nodes, u.elem_nodes)])
    ref, _ = orc.laplace_assemble(u.elem_nodes, u.coords, rp, ci)
    assert np.linalg.norm(eq.matrix_values() - ref) <= 1e-12 * np.linalg.norm(ref)
    for fixed in (boundary, np.concatenate([[0], boundary, [u.n_nodes - 1]])):
        eq.set_boundary_conditions(fixed, field[fixed])
        for _ in range(2):
            check_restriction(eq, fixed, cm.OC_FP64)
        eq.solve(cm.newton_options(krylov_relative_tolerance=1e-12, absolute_tolerance=0.0))
        want = field.copy()
        want[np.setdiff1d([0, u.n_nodes - 1], fixed)] = 0.0
        assert np.linalg.norm(eq.get_dofs() - want) < 8e-9 * np.linalg.norm(want)
    eq.destroy()
