"""The V-cycle whose first post-smoothing sweep reads A P0 (the Jacobian times
the trilinear interpolation) against the same V-cycle with every level-0 sweep
a pass over the Jacobian: equal linear operators, so GMRES needs the same
iterations.  The counts below are the latter's, on the smallest meshes (one
element: every neighbour box clipped; odd and even coarse grids) and over the
sweep options with and without post-smoothing.  Rounding may move the stopping
test by one iteration per Newton step, no more; a wrong product, slot or mask
costs tens."""
import pytest

pytestmark = pytest.mark.gpu

# (pre, post): GMRES iterations to rtol 1e-8 for n = 1, 2, 3, 5
COUNTS = {(1, 2): (60, 124, 173, 219), (2, 1): (62, 126, 173, 219), (1, 0): (83, 161, 237, 306),
          (2, 3): (53, 111, 155, 192)}


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("k,n", list(enumerate((1, 2, 3, 5))))
@pytest.mark.parametrize("pre,post", list(COUNTS))
def test_krylov_iterations_of_the_full_pass_cycle(gpu, pre, post, k, n, precision):
    cm = gpu
    mesh = cm.RegularMesh.generate(2, n, jitter=0.1, seed=40 + n)
    eq = cm.MooneyRivlinEquationsSet(mesh, 2.0, 6.0)
    eq.set_dofs(eq.undeformed_dofs())
    eq.uniaxial_boundary_conditions(1.1)
    eq.set_multigrid(pre, post, 0.6)
    eq.load_increment_apply(1, 4)
    st = eq.newton_solve(cm.newton_options(solution_tolerance=0.0, relative_tolerance=1e-10, absolute_tolerance=0.0,
                                           krylov_restart=100, krylov_relative_tolerance=1e-8, fallback=0,
                                           jacobian_precision=precision, maximum_iterations=30,
                                           preconditioner=cm.OC_PRECONDITIONER_MULTIGRID))
    eq.destroy()
    assert st["converged"], st
    assert abs(st["krylov_iterations"] - COUNTS[pre, post][k]) <= st["newton_iterations"]


def test_sweep_options_changed_after_a_solve(gpu):
    """The stencil levels' composed maps hold omega: a solve after
    oc_multigrid_options_set is the one a fresh set with those options makes."""
    cm = gpu
    opts = cm.newton_options(solution_tolerance=0.0, relative_tolerance=1e-10, absolute_tolerance=0.0,
                             krylov_restart=100, krylov_relative_tolerance=1e-8, fallback=0,
                             preconditioner=cm.OC_PRECONDITIONER_MULTIGRID)
    out = []
    for first in (0.9, None):
        mesh = cm.RegularMesh.generate(2, 5, jitter=0.1, seed=45)
        eq = cm.MooneyRivlinEquationsSet(mesh, 2.0, 6.0)
        eq.uniaxial_boundary_conditions(1.1)
        eq.set_multigrid(1, 2, first or 0.6)
        if first:
            eq.set_dofs(eq.undeformed_dofs())
            eq.load_increment_apply(1, 4)
            eq.newton_solve(opts)
            cm._lib.call("oc_multigrid_options_set", eq.handle, 1, 2, 0.6)
        eq.set_dofs(eq.undeformed_dofs())
        eq.load_increment_apply(1, 4)
        st = eq.newton_solve(opts)
        out.append((st["krylov_iterations"], eq.get_dofs()))
        eq.destroy()
    assert out[0][0] == out[1][0]
    assert (out[0][1] == out[1][1]).all()
