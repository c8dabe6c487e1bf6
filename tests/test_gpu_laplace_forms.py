"""The three forms of the Laplace assembly (one launch on small meshes, element
buffer and row gather, fused structured grid) at the sizes where they change and
where their blocks end."""
import numpy as np
import pytest

import oracle_lib as orc

pytestmark = pytest.mark.gpu


def _check(cm, mesh, fused):
    eq = cm.LaplaceEquationsSet(mesh)
    assert bool(eq.set_fused(fused)) == (fused == 2)
    eq.assemble()
    rp, ci = eq.matrix_structure(0)
    ovals, _ = orc.laplace_assemble(mesh.elem_nodes, mesh.coords, rp.astype(np.int64), ci)
    vals = eq.matrix_values()
    assert np.linalg.norm(vals - ovals) < 1e-12 * np.linalg.norm(ovals)  # the parity tests' bound
    assert np.array_equal(eq.rhs(), np.zeros(eq.n_rows))


# one row block of eight and its remainders; the last size of the one-launch
# form (11,913 rows) and the first of the two passes (12,144); 64-element blocks
# with a remainder.  User numbering: no order to rely on.
@pytest.mark.parametrize("n", [(1, 1, 1), (2, 1, 3), (7, 5, 3), (18, 18, 32), (21, 22, 23), (24, 23, 22)])
def test_passes(gpu, n):
    mesh = gpu.RegularMesh.generate(1, n, jitter=0.15, seed=5)
    order = np.random.default_rng(1).permutation(mesh.n_nodes)
    _check(gpu, gpu.as_user_mesh(mesh, region_order=order), 0)


# node columns of 15 x 7: one short of a tile, a whole one, one over; one and
# two layers; a grid of the four- and of the eight-layer segments
@pytest.mark.parametrize("n", [(13, 5, 1), (14, 6, 2), (15, 7, 3), (30, 13, 5), (1, 50, 2), (64, 64, 40), (80, 80, 64)])
def test_fused(gpu, n):
    _check(gpu, gpu.RegularMesh.generate(1, n, jitter=0.15, seed=6), 2)
