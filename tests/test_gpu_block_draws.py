"""The block sweeps' workgroups draw their blocks: each takes several (grids far
below the number of blocks), and several matrices' sweeps run side by side with
more workgroups than the GPU holds at once.  Bitwise against the oracle, or
against the same solve alone."""
import threading

import numpy as np
import pytest

from test_gpu_blocks import nine_point
from tflows_amd import mesh

pytestmark = pytest.mark.gpu


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


SYSTEMS = {"33x16x25": lambda: box(33, 16, 25), "61x40x23": lambda: box(61, 40, 23),
           "nine33x70": lambda: nine_point(33, 70)}


@pytest.mark.parametrize("groups", [1, 3, 7])
@pytest.mark.parametrize("name", SYSTEMS)
def test_several_blocks_each(S, oracle, monkeypatch, name, groups):
    import torch
    row, col, dia, val, b = SYSTEMS[name]()
    print(f"block draws {name} groups={groups}", flush=True)
    monkeypatch.setenv("TFS_SWEEP_GROUPS", str(groups))
    A = S.Matrix(row, col, dia, val)
    nblk = mesh.layout_blocks(row, col, dia)[0]
    assert A.info()["sweep_groups"] == groups < nblk
    d_or = oracle.prec_form(row, col, dia, val, 2)
    z_or = oracle.prec_solve(row, col, dia, val, d_or, 2, b)
    db = torch.from_numpy(b).cuda()
    d, z = torch.zeros_like(db), torch.zeros_like(db)
    for scale in (1.0, 1.0, 2.0):
        A.set_values(scale * val)
        A.prec_form(2)
        A.prec_diag(d)
        assert np.array_equal(d.cpu().numpy(), oracle.prec_form(row, col, dia, scale * val, 2))
        for _ in range(3 if scale == 1.0 else 0):
            z.zero_()
            A.prec_solve(2, db, z)
            assert np.array_equal(z.cpu().numpy(), z_or)
    # a solve queues iterations past its end: their sweeps find it done and leave
    A.set_values(val)
    tol = 1e-10 * float(np.linalg.norm(b))
    ref = oracle.solve("cg", row, col, dia, val, b, prec=2, niter=2000, tol=tol)
    for _ in range(2):
        x, r = torch.zeros_like(db), db.clone()
        n, _, _ = S.solve("cg", A, x, r, 2, 2000, tol)
        assert abs(n - ref["niter"]) <= max(1, ref["niter"] // 20)
        z.zero_()
        A.prec_solve(2, db, z)
        assert np.array_equal(z.cpu().numpy(), z_or)


def test_many_matrices_at_once(S):
    """Seven solves from seven threads, their grids together more than the GPU
    holds: each ends, with the bits it gives alone."""
    import torch
    systems = [box(65, 57, 61), box(97, 75, 61), nine_point(400, 300), box(64, 64, 64),
               box(97, 75, 61), nine_point(300, 500), box(65, 57, 61)]
    cases = []
    for row, col, dia, val, b in systems:
        A = S.Matrix(row, col, dia, val)
        cases.append((A, torch.from_numpy(b).cuda(), 1e-6 * float(np.linalg.norm(b))))
    groups = sum(A.info()["sweep_groups"] for A, _, _ in cases)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert groups > 5 * cus   # at most five (narrow) or three (wide) of them on a CU
    torch.cuda.synchronize()

    def run(i, out):
        A, b, tol = cases[i]
        x, r = torch.zeros_like(b), b.clone()
        torch.cuda.synchronize()
        out[i] = S.solve("cg", A, x, r, 2, 60, tol) + (x.cpu().numpy(),)

    alone, beside = {}, {}
    for i in range(len(cases)):
        print("alone", i, flush=True)
        run(i, alone)
    for rnd in range(2):
        print("side by side", rnd, flush=True)
        threads = [threading.Thread(target=run, args=(i, beside)) for i in range(len(cases))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        for i in range(len(cases)):
            assert alone[i][:3] == beside[i][:3]
            assert np.array_equal(alone[i][3], beside[i][3])
