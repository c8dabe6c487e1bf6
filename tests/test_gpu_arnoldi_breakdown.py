"""The Arnoldi process past the end of its Krylov space, where a new vector is
rounding alone and its second Gram-Schmidt pass cancels like the first: its norm
must be that of the vector, not a difference of rounding, which comes out as zero
about every second time and ends the cycle as solved.  With a tolerance of zero one
cycle then runs to the iteration limit, accurate all along, and a restarted solve
past its first cycle (it may end once the true residual is zero)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 2 to 36 free nodes of small meshes (one row a thread, up to 32 vectors and more),
# restarts below, at and above their number, and clusters of them in meshes of the
# 512- and 1,024-thread blocks.  The residual is rounding (below 1e-14 of the right
# side) and the condition number below 3 N^2 for N elements across the free nodes.
@pytest.mark.parametrize("n,restart", [((3, 2, 2), 60), ((3, 3, 2), 60), ((3, 3, 3), 8), ((3, 3, 3), 60), ((4, 4, 3), 17),
                                       ((4, 4, 3), 60), ((5, 4, 4), 36), ((5, 4, 4), 60)])
@pytest.mark.parametrize("around", [0, 20, 25])
def test_zero_tolerance(gpu, n, restart, around):
    cm = gpu
    limit = 60
    big = tuple(k + 2 * around for k in n)
    mesh = cm.RegularMesh.generate(1, big, jitter=0.1, seed=2)
    u = np.array([0.4, 0.2, -0.9]) @ mesh.coords - 0.3
    g = np.stack(np.unravel_index(np.arange(mesh.n_nodes), tuple(k + 1 for k in big), order="F"))
    inner = np.all([(g[a] > around) & (g[a] < around + n[a]) for a in range(3)], axis=0)
    fixed = np.nonzero(~inner)[0]
    assert mesh.n_nodes - len(fixed) == np.prod([k - 1 for k in n])
    eq = cm.LaplaceEquationsSet(mesh)
    eq.set_boundary_conditions(fixed, u[fixed])
    st = eq.solve(cm.newton_options(krylov_relative_tolerance=0.0, absolute_tolerance=0.0, krylov_restart=restart,
                                    krylov_maximum_iterations=limit), raise_on_failure=False)
    assert st["krylov_iterations"] == limit if restart == limit else st["krylov_iterations"] > restart, st
    assert np.linalg.norm((eq.get_dofs() - u)[inner]) < 3 * max(n) ** 2 * 1e-14 * np.linalg.norm(u[inner])
    eq.destroy()


@pytest.mark.parametrize("seed", [1, 2, 3, 4])
def test_inconsistent_system_is_not_solved(gpu, seed):
    """One element with its centre node free: three displacements cannot meet eight
    pressure equations, so no linear solve may end within its tolerance."""
    cm = gpu
    mesh = cm.RegularMesh.generate(2, 1, jitter=0.1, seed=seed)
    eq = cm.MooneyRivlinEquationsSet(mesh, 2.0, 6.0)
    d = eq.undeformed_dofs() * 1.02
    eq.set_dofs(d)
    fixed = np.setdiff1d(np.arange(81), [13, 40, 67])
    eq.set_boundary_conditions(fixed, d[fixed])
    st = eq.newton_solve(cm.newton_options(krylov_relative_tolerance=1e-10, krylov_restart=40,
                                           krylov_maximum_iterations=80, maximum_iterations=3,
                                           preconditioner=cm.OC_PRECONDITIONER_BLOCK_DIAGONAL), raise_on_failure=False)
    assert st["reason"] == cm.OC_DIVERGED_LINEAR_SOLVE, st
    eq.destroy()
