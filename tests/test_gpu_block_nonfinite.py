"""Infinities and NaN through the block sweeps (whose waiting values are a NaN
pattern) and the brick sweeps: the values of one launch per level, and the solve's
own end."""
import numpy as np
import pytest

from test_gpu_blocks import nine_point
from tflows_amd import mesh

pytestmark = pytest.mark.gpu

SENTINEL = np.uint64(0xFFF4DEADBEEFC0DE)   # what an output holds until it is formed


@pytest.fixture(scope="module")
def S():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no GPU visible")
    from tflows_amd import solvers
    return solvers


def box(*d):
    c = mesh.make_case(kind=mesh.POISSON, nx=d[0], ny=d[1], nz=d[2], beta=1.0)
    return c.row, c.col, c.dia, c.val, c.b


@pytest.mark.parametrize("system", [lambda: box(33, 16, 25), lambda: nine_point(33, 70)])
@pytest.mark.parametrize("where", ["first", "middle", "all"])
def test_blocks(S, system, where):
    import torch
    row, col, dia, val, b = system()
    n = len(b)
    for bits in (np.inf, -np.inf, np.nan, SENTINEL):
        b = b.copy()
        at = {"first": [0], "middle": [n // 2, n // 2 + 7], "all": slice(None)}[where]
        if isinstance(bits, np.uint64):
            b.view(np.uint64)[at] = bits
        else:
            b[at] = bits
        print(f"nonfinite {where} {bits} n={n}", flush=True)
        A = S.Matrix(row, col, dia, val)
        db = torch.from_numpy(b).cuda()
        z = [torch.zeros_like(db) for _ in range(2)]
        A.prec_form(2)
        A.prec_solve(2, db, z[0])
        A.set_sweep_schedule(S.TFS_SWEEP_LEVELS)
        A.prec_solve(2, db, z[1])
        u, w = (t.cpu().numpy() for t in z)
        assert np.isnan(u).any() or np.isinf(u).any()
        assert np.array_equal(u, w, equal_nan=True)
        A.close()


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_bricks(S, bad):
    import torch
    row, col, dia, val, b = box(40, 40, 40)
    b = b.copy()
    b[12345] = bad
    ends = []
    for schedule in (S.TFS_SWEEP_STATIC, S.TFS_SWEEP_LEVELS):
        A = S.Matrix(row, col, dia, val)
        A.set_inner_order(S.TFS_INNER_BRICKS)
        A.set_sweep_schedule(schedule)
        x, r = torch.zeros(len(b), dtype=torch.float64, device="cuda"), torch.from_numpy(b).cuda()
        print(f"bricks {bad} schedule {schedule}", flush=True)
        try:
            ends.append(("ok", S.solve_mixed(A, x, r, 2, 200, 1e-6)[0]))
        except S.SolverError as e:
            ends.append(("error", e.status))
        A.close()
    assert ends[0] == ends[1]
