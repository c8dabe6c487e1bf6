"""The FP64 product of a wavefront per node on meshes that no regular grid has:
nodes of five elements around an axis (155 neighbours, more than two rounds of the
wavefront, and 498 entries of the 504 a row may have), and three elements over the
same nodes with pressures of their own (81 pressure columns, more than one round).
As in test_gpu_flat_rows, Newton with the block preconditioner must converge
quadratically to the oracle's residual tolerance."""
import numpy as np
import pytest

import oracle_lib as orc
from cm_amd.mesh import RegularMesh, UserMesh

pytestmark = pytest.mark.gpu


def around_an_axis(k, layers):
    """k quadrilaterals around the z axis, extruded; nodes user-numbered by position."""
    def ray(i, r):
        return np.array([r * np.cos(2 * np.pi * i / k), r * np.sin(2 * np.pi * i / k)])
    points = []
    for layer in range(layers):
        for i in range(k):
            c = [np.zeros(2), ray(i, 1.0), ray(i + 1, 1.0), ray(i + 0.5, 1.3)]
            for z in (0.0, 0.5, 1.0):
                for y in (0.0, 0.5, 1.0):
                    for x in (0.0, 0.5, 1.0):
                        p = (1 - x) * (1 - y) * c[0] + x * (1 - y) * c[1] + (1 - x) * y * c[2] + x * y * c[3]
                        points.append((p[0], p[1], layer + z))
    points = np.array(points)
    _, index, nodes = np.unique(np.round(points, 6), axis=0, return_index=True, return_inverse=True)
    nodes = nodes.reshape(-1, 27)
    return UserMesh.from_user_numbers(2, np.arange(index.size), points[index].T, nodes,
                                      nodes[:, [0, 2, 6, 8, 18, 20, 24, 26]])


def copies(m, count):
    """The elements of a mesh `count` times over the same nodes, with pressure nodes of their own."""
    u = UserMesh(2, np.tile(m.elem_nodes, (count, 1)), m.coords, np.arange(m.n_nodes))
    u.elem_nodes_l = np.concatenate([m.elem_nodes_l + i * m.n_nodes_l for i in range(count)]).astype(np.int32)
    u.node_user_numbers_l = np.arange(count * m.n_nodes_l)
    return u


@pytest.mark.parametrize("name,longest", [("axis", 498), ("copies", 3 * 125 + 81)])
def test_newton_by_the_wavefront_product(gpu, name, longest):
    cm = gpu
    mesh = around_an_axis(5, 2) if name == "axis" else copies(RegularMesh.generate(2, 2, jitter=0.1, seed=4), 3)
    eq = cm.MooneyRivlinEquationsSet(mesh, 2.0, 6.0)
    assert np.diff(eq.matrix_structure()[0]).max() == longest
    eq.set_dofs(eq.undeformed_dofs())
    # the bottom held, the top pulled up by 3%, free sideways
    nq, z = mesh.n_nodes, mesh.coords[2]
    bottom, top = mesh.coords.min(axis=1)[2] == z, mesh.coords.max(axis=1)[2] == z
    b, t = np.nonzero(bottom)[0], np.nonzero(top)[0]
    fixed = np.concatenate([b, nq + b, 2 * nq + b, 2 * nq + t])
    values = np.concatenate([mesh.coords[:, b].ravel(), z[t] + 0.03 * (z.max() - z.min())])
    eq.set_boundary_conditions(fixed, values)
    eq.load_increment_apply(1, 1)
    ref = eq.residual_norm()
    st = eq.newton_solve(cm.newton_options(solution_tolerance=0.0, relative_tolerance=1e-10, absolute_tolerance=0.0,
                                           krylov_restart=300, krylov_relative_tolerance=1e-9,
                                           preconditioner=cm.OC_PRECONDITIONER_BLOCK_TRIANGULAR,
                                           maximum_iterations=12))
    assert st["converged"] and st["newton_iterations"] <= 7, st
    r = orc.mr_residual(mesh.elem_nodes, mesh.elem_nodes_l, mesh.coords, eq.get_dofs(), 2.0, 6.0)
    r[fixed] = 0.0
    assert np.linalg.norm(r) <= 1.05e-10 * ref
    eq.destroy()
