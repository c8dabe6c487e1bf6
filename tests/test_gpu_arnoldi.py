"""The Arnoldi process of the GMRES solver at the edges of its launch shapes:
one row, a block's last rows, the sizes at which the blocks grow from 256 to 512
and 1,024 threads, and restarts around the eight vectors a block takes at once."""
import numpy as np
import pytest

import cm_amd as cm

pytestmark = pytest.mark.gpu


def _solve(n, **options):
    """A linear field (in the trilinear space, so the exact solution) from its boundary values."""
    cm.initialise(0)
    mesh = cm.RegularMesh.generate(1, n, jitter=0.1, seed=3)
    u = np.array([0.3, -0.7, 0.2]) @ mesh.coords + 0.1
    boundary = np.unique(np.concatenate([mesh.face_nodes(a, side) for a in range(3) for side in (0, 1)]))
    eq = cm.LaplaceEquationsSet(mesh)
    eq.set_boundary_conditions(boundary, u[boundary])
    eq.solve(cm.newton_options(krylov_relative_tolerance=1e-12, absolute_tolerance=0.0, **options))
    return np.linalg.norm(eq.get_dofs() - u) / np.linalg.norm(u)


# 27 rows (one free), 125, 256-row edges, then the 512- and 1,024-thread blocks
# (over 65,536 and over 131,072 rows).  The relative residual of 1e-12 times the
# matrix's condition number, below 3 N^2 for N elements per direction and 0.1 h
# jitter, bounds the error: under 8e-9 at 51 elements.
@pytest.mark.parametrize("n", [(2, 2, 2), (4, 4, 4), (7, 7, 3), (15, 3, 3), (40, 40, 39), (51, 51, 50)])
def test_launch_shapes(n):
    assert _solve(n) < 8e-9


# the restart bounds the vectors of a step: 1 to 40 of them, across multiples of eight
@pytest.mark.parametrize("restart", [3, 6, 7, 8, 15, 16, 40, 200])
def test_restarts(restart):
    assert _solve((9, 8, 7), krylov_restart=restart) < 8e-9
