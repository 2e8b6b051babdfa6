"""spmv and residual on the caller's own rows (numberings that gather well)
and through the S order (the others, and x overlapping y): bitwise the oracle's
row sums, at the edges of a row block, with rows longer than one, in place."""
import numpy as np
import pytest

from tflows_amd import mesh

pytestmark = pytest.mark.gpu


def box(permute, *d):
    c = mesh.make_case(nx=d[0], ny=d[1], nz=d[2], permute=permute)
    return c.row, c.col, c.dia, c.val


def arrow(n, every):
    """Diagonal plus a full first row and column: one row longer than a row block."""
    rows = [np.arange(n)] + [np.array([0, i]) if i % every == 0 else np.array([i])
                             for i in range(1, n)]
    row = np.concatenate(([0], np.cumsum([len(r) for r in rows]))).astype(np.int32)
    col = np.concatenate(rows).astype(np.int32)
    dia = np.array([row[i] + int(np.searchsorted(rows[i], i)) for i in range(n)], np.int32)
    return row, col, dia, np.random.default_rng(3).standard_normal(len(col))


CASES = {
    "one": lambda: box(False, 1, 1, 1), "63": lambda: box(False, 7, 9, 1),
    "64": lambda: box(False, 4, 4, 4), "65": lambda: box(False, 13, 5, 1),
    "box": lambda: box(False, 37, 29, 41), "permuted": lambda: box(True, 37, 29, 41),
    "arrow": lambda: arrow(1500, 1), "sparse arrow": lambda: arrow(4000, 7),
}


@pytest.mark.parametrize("name", CASES)
def test_products(oracle, name):
    import torch
    from tflows_amd import solvers
    row, col, dia, val = CASES[name]()
    n = len(row) - 1
    print(f"products {name} n={n}", flush=True)
    A = solvers.Matrix(row, col, dia, val)
    u = np.random.default_rng(n)
    buf = torch.from_numpy(u.uniform(-1, 1, 2 * n)).cuda()
    h = buf.cpu().numpy()
    for x0, y0 in ((0, n), (n, 0), (0, 0), (0, n // 2)):   # apart, and overlapping
        b = buf.clone()
        x, y = b[x0:x0 + n], b[y0:y0 + n]
        A.residual(x, y)
        assert np.array_equal(y.cpu().numpy(),
                              oracle.residual(row, col, dia, val, h[x0:x0 + n], h[y0:y0 + n]))
        b = buf.clone()
        x, y = b[x0:x0 + n], b[y0:y0 + n]
        A.spmv(x, y)
        assert np.array_equal(y.cpu().numpy(), oracle.spmv(row, col, dia, val, h[x0:x0 + n]))
