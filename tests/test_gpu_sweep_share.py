"""The row-by-row FP64 sweeps fit six workgroups on every CU, of which the server's
concurrent sweeps each get a share."""
import numpy as np
import pytest

from tflows_amd import mesh

pytestmark = pytest.mark.gpu


def test_workgroups_that_fit(oracle, monkeypatch):
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no GPU visible")
    from tflows_amd import solvers as S
    c = mesh.make_case(kind=mesh.MOMENTUM, nx=75, beta=2.0, jitter=0.1, permute=True,
                       pin_first=False, rhs_zero_mean=False)
    monkeypatch.setenv("TFS_SWEEP_GROUPS", "100000")   # the cap: what fits at once
    A = S.Matrix(c.row, c.col, c.dia, c.val)
    want = 6 * torch.cuda.get_device_properties(0).multi_processor_count
    assert (c.n + 255) // 256 >= want
    assert A.info()["sweep_groups"] >= want
    A.set_sweep_schedule(S.TFS_SWEEP_STATIC)
    # and with all of them the sweeps are the reference's
    d_or = oracle.prec_form(c.row, c.col, c.dia, c.val, 2)
    z_or = oracle.prec_solve(c.row, c.col, c.dia, c.val, d_or, 2, c.b)
    db = torch.from_numpy(c.b).cuda()
    z = torch.empty_like(db)
    A.prec_form(2)
    A.prec_solve(2, db, z)
    assert np.array_equal(z.cpu().numpy(), z_or)
