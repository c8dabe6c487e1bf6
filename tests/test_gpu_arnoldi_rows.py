"""The Arnoldi step with the dot products in the SpMV's launch and one row a
thread: a block's 128 rows exactly and one plane more, 32,768 rows (the most it
takes) and the next grid, and restarts at the 32 vectors a row keeps in
registers.  Bound as in test_gpu_arnoldi: 1e-12 times a condition number below
3 N^2."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,restart", [((3, 3, 7), 30), ((3, 3, 8), 30), ((31, 31, 31), 30), ((32, 31, 31), 30),
                                       ((12, 11, 10), 29), ((12, 11, 10), 31), ((12, 11, 10), 33)])
def test_linear_field(gpu, n, restart):
    cm = gpu
    mesh = cm.RegularMesh.generate(1, n, jitter=0.1, seed=5)
    u = np.array([0.4, 0.2, -0.9]) @ mesh.coords - 0.3
    boundary = np.unique(np.concatenate([mesh.face_nodes(a, side) for a in range(3) for side in (0, 1)]))
    eq = cm.LaplaceEquationsSet(mesh)
    eq.set_boundary_conditions(boundary, u[boundary])
    eq.solve(cm.newton_options(krylov_relative_tolerance=1e-12, absolute_tolerance=0.0, krylov_restart=restart))
    assert np.linalg.norm(eq.get_dofs() - u) / np.linalg.norm(u) < 3 * max(n) ** 2 * 1e-12
    eq.destroy()
