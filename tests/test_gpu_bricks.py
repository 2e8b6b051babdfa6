"""The FP32 sweeps of a two-coloured brick copy (one wavefront per unit of
bricks), bitwise against the level-by-level schedule of the same copy, where
they can go wrong: boxes at and around whole bricks, thin ones (merged units,
bricks of one row per step), odd remainders, and a schedule changed on a formed
copy and back, with new values in between."""
import numpy as np
import pytest

from tflows_amd import mesh

pytestmark = pytest.mark.gpu

BOXES = [(16, 16, 16), (32, 32, 32), (33, 17, 40), (47, 31, 16), (2, 3, 400), (90, 1, 70),
         (12, 9, 7), (1, 1, 500), (65, 48, 34)]


@pytest.fixture(scope="module")
def torch():
    import torch as t
    if not t.cuda.is_available():
        pytest.fail("no GPU visible")
    return t


@pytest.mark.parametrize("dims", BOXES, ids=lambda d: "x".join(map(str, d)))
def test_brick_sweeps_bitwise(torch, dims):
    from tflows_amd import solvers as S
    c = mesh.make_case(kind=mesh.POISSON, nx=dims[0], ny=dims[1], nz=dims[2], beta=1.0)
    tol = 1e-10 * float(np.linalg.norm(c.b))
    print(f"bricks {dims} n={c.n}", flush=True)

    def solve(A):
        x = torch.zeros(c.n, dtype=torch.float64, device="cuda")
        r = torch.from_numpy(c.b.copy()).cuda()
        out = S.solve_mixed(A, x, r, 2, 20, tol)
        return out, x.cpu().numpy()

    A = S.Matrix(c.row, c.col, c.dia, c.val)
    A.set_inner_order(S.TFS_INNER_BRICKS)
    B = S.Matrix(c.row, c.col, c.dia, c.val)
    B.set_inner_order(S.TFS_INNER_BRICKS)
    B.set_sweep_schedule(S.TFS_SWEEP_LEVELS)
    want, xw = solve(B)
    got, xg = solve(A)
    colours = A.info()["inner_colours"]
    print("colours", colours, flush=True)
    assert colours == 2 or any(d % 16 for d in dims)  # (ragged bricks may need more)
    assert got == want and np.array_equal(xg, xw)
    # the copy's sweeps leave the bricks and come back, with new values
    for schedule in (S.TFS_SWEEP_DYNAMIC, S.TFS_SWEEP_STATIC, S.TFS_SWEEP_LEVELS):
        scaled = c.val.copy()
        scaled[c.dia] *= 1.0 + 0.01 * (schedule + 1)
        for M in (A, B):
            M.set_values(scaled)
        A.set_sweep_schedule(schedule)
        want, xw = solve(B)
        got, xg = solve(A)
        assert got == want and np.array_equal(xg, xw)
