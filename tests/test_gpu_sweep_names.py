"""tfs_matrix_sweep_kernel names the kernel that the sweeps run."""
import numpy as np
import pytest

from tflows_amd import mesh

pytestmark = pytest.mark.gpu


def test_names():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no GPU visible")
    from tflows_amd import solvers as S
    c = mesh.make_case(nx=24, beta=1.0)

    def refined(order):
        A = S.Matrix(c.row, c.col, c.dia, c.val)
        A.set_inner_order(order)
        x, r = torch.zeros(c.n, dtype=torch.float64, device="cuda"), torch.from_numpy(c.b).cuda()
        S.solve_mixed(A, x, r, 2, 200, 1e-6 * float(np.linalg.norm(c.b)))
        return A

    A = S.Matrix(c.row, c.col, c.dia, c.val)
    assert A.sweep_kernel() == "k_block_sweep" and A.sweep_kernel(inner=True) == ""
    A.set_sweep_schedule(S.TFS_SWEEP_LEVELS)
    assert A.sweep_kernel() == "k_level"
    A.set_sweep_schedule(S.TFS_SWEEP_DYNAMIC)
    assert A.sweep_kernel() == "k_sweep_syncfree"
    assert refined(S.TFS_INNER_BRICKS).sweep_kernel(inner=True) == "k_brick_sweep"
    assert refined(S.TFS_INNER_COLOURED).sweep_kernel(inner=True) == "k_colour_sweep"
    B = refined(S.TFS_INNER_BRICKS)
    B.set_sweep_schedule(S.TFS_SWEEP_LEVELS)
    assert B.sweep_kernel(inner=True) == "k_level"
