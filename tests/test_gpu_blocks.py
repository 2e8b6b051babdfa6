"""The FP64 factor and sweeps over row blocks (one wavefront per block),
bitwise against the oracle, where they can go wrong: boxes smaller than, equal
to and just beyond one block, thin and ragged ones, blocks of odd row counts,
rows with more than three entries in a triangle (the wide kernel), chains
(blocks of one row per step), and a schedule changed on a formed factor."""
import numpy as np
import pytest

from tflows_amd import mesh

pytestmark = pytest.mark.gpu

BOXES = [(8, 8, 8), (9, 8, 8), (9, 17, 7), (33, 16, 25), (2, 3, 200), (30, 1, 40), (1, 1, 700),
         (25, 25, 25), (61, 40, 23)]


@pytest.fixture(scope="module")
def torch():
    import torch as t
    if not t.cuda.is_available():
        pytest.fail("no GPU visible")
    return t


def nine_point(nx, ny, seed=3):
    """A 9-point stencil on an nx x ny grid (four lower entries per row)."""
    row, col, dia = [0], [], []
    for i in range(nx * ny):
        x, y = i % nx, i // nx
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                if 0 <= x + dx < nx and 0 <= y + dy < ny:
                    if dx == dy == 0:
                        dia.append(len(col))
                    col.append(i + dx + dy * nx)
        row.append(len(col))
    rng = np.random.default_rng(seed)
    val = -rng.uniform(0.5, 1.0, len(col))
    val[dia] = 9.0
    return (np.array(row, np.int32), np.array(col, np.int32), np.array(dia, np.int32), val,
            rng.uniform(-1.0, 1.0, nx * ny))


def systems():
    for d in BOXES:
        c = mesh.make_case(kind=mesh.POISSON, nx=d[0], ny=d[1], nz=d[2], beta=1.0)
        yield "x".join(map(str, d)), (c.row, c.col, c.dia, c.val, c.b)
    for d in ((40, 9), (33, 70)):
        yield f"nine{d[0]}x{d[1]}", nine_point(*d)


@pytest.mark.parametrize("name,system", list(systems()), ids=lambda v: v if isinstance(v, str)
                         else "")
def test_block_sweeps_bitwise(torch, oracle, name, system):
    from tflows_amd import solvers as S
    row, col, dia, val, b = system
    n = len(b)
    print(f"blocks {name} n={n}", flush=True)
    A = S.Matrix(row, col, dia, val)
    d_or = oracle.prec_form(row, col, dia, val, 2)
    z_or = oracle.prec_solve(row, col, dia, val, d_or, 2, b)
    db = torch.from_numpy(b).cuda()
    d, z = torch.zeros_like(db), torch.zeros_like(db)
    A.prec_form(2)
    for schedule in (None, S.TFS_SWEEP_STATIC, S.TFS_SWEEP_LEVELS, S.TFS_SWEEP_STATIC,
                     S.TFS_SWEEP_DYNAMIC, S.TFS_SWEEP_STATIC):
        if schedule is not None:
            A.set_sweep_schedule(schedule)
        for _ in range(2):
            z.zero_()
            A.prec_solve(2, db, z)
            assert np.array_equal(z.cpu().numpy(), z_or), schedule
        A.prec_diag(d)
        assert np.array_equal(d.cpu().numpy(), d_or), schedule
    # new values through the same layouts
    A.set_values(2.0 * val)
    A.prec_form(2)
    A.prec_diag(d)
    assert np.array_equal(d.cpu().numpy(), oracle.prec_form(row, col, dia, 2.0 * val, 2))
