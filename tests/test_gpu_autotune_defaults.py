"""What the launch-shape autotuner keeps: a shape replaces the default that the
launch itself would pick for this mesh and precision, and only there."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = {"element_matrix_ms": lambda c: str(c["element_blocks_per_cu"]), "row_gather_ms": lambda c: str(c["gather_chunk"]),
          "spmv_ms": lambda c: f"{c['spmv_lanes']}x{c['spmv_unroll']}"}


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,gather", [(2, 8), (8, 4)])  # 152 and 5,642 nodes; eight element rows up to 8 a CU
def test_choice_against_the_launch_default(gpu, n, gather, precision):
    cm = gpu
    eq = cm.MooneyRivlinEquationsSet(cm.RegularMesh.generate(2, n, jitter=0.1, seed=5), 2.0, 6.0)
    eq.set_dofs(eq.undeformed_dofs())
    r = eq.autotune(precision)
    assert r["default"]["gather_chunk"] == gather
    assert (r["default"]["spmv_lanes"], r["default"]["spmv_unroll"]) == ((32, 2) if precision else (64, 1))
    for times, key in SHAPES.items():
        chosen, default = key(r["chosen"]), key(r["default"])
        # the report gives times in 0.1 us
        assert chosen == default or r[times][chosen] <= (1 - r["margin"]) * r[times][default] + 1e-4, (times, r)
    eq.destroy()


@pytest.mark.parametrize("tuned,solved", [(0, 1), (1, 0)])
@pytest.mark.parametrize("multigrid", [False, True])
def test_other_precision_keeps_its_defaults(gpu, tuned, solved, multigrid):
    """Sums run in another order in another shape: solutions equal bit for bit
    show that the launches of one precision ignore what was tuned for the other."""
    cm = gpu
    results = []
    for tune in (False, True):
        eq = cm.MooneyRivlinEquationsSet(cm.RegularMesh.generate(2, 4, jitter=0.1, seed=5), 2.0, 6.0)
        eq.set_dofs(eq.undeformed_dofs())
        if tune:
            eq.autotune(tuned)
        eq.uniaxial_boundary_conditions(1.05)
        if multigrid:
            eq.set_multigrid()
        eq.load_increment_apply(1, 1)
        eq.newton_solve(cm.newton_options(
            solution_tolerance=0.0, relative_tolerance=1e-8, krylov_restart=100, krylov_relative_tolerance=1e-4,
            jacobian_precision=solved,
            preconditioner=cm.OC_PRECONDITIONER_MULTIGRID if multigrid else cm.OC_PRECONDITIONER_BLOCK_TRIANGULAR))
        results.append(eq.get_dofs())
        eq.destroy()
    assert np.array_equal(results[0], results[1])
