"""The FP64 product of a wavefront per node (columns read once, values in
16-byte loads at each row's own shift): Newton with the block preconditioner,
whose only matrix product it is, must converge quadratically to the oracle's
residual tolerance on meshes whose rows start at every shift and whose nodes
have from 27 (one element) to 125 neighbours."""
import numpy as np
import pytest

import oracle_lib as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1, 1, 1), (2, 1, 1), (1, 3, 2), (3, 2, 5)])
def test_newton_by_the_wavefront_product(gpu, n):
    cm = gpu
    mesh = cm.RegularMesh.generate(2, n, jitter=0.1, seed=sum(n))
    eq = cm.MooneyRivlinEquationsSet(mesh, 2.0, 6.0)
    eq.set_dofs(eq.undeformed_dofs())
    fixed = eq.uniaxial_boundary_conditions(1.05)
    eq.load_increment_apply(1, 1)
    ref = eq.residual_norm()
    st = eq.newton_solve(cm.newton_options(solution_tolerance=0.0, relative_tolerance=1e-10, absolute_tolerance=0.0,
                                           krylov_restart=200, krylov_relative_tolerance=1e-9,
                                           preconditioner=cm.OC_PRECONDITIONER_BLOCK_TRIANGULAR,
                                           maximum_iterations=12))
    assert st["converged"] and st["newton_iterations"] <= 7, st
    r = orc.mr_residual(mesh.elem_nodes, mesh.elem_nodes_l, mesh.coords, eq.get_dofs(), 2.0, 6.0)
    r[fixed] = 0.0
    assert np.linalg.norm(r) <= 1.05e-10 * ref
    eq.destroy()
