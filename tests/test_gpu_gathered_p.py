"""CG forms its search direction in the product where rows are short and in a
pass of its own where they are wide (more than 20 entries on average), which
shows in the work vectors it holds (the former needs one more); both against
the oracle."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def band(n, entries, seed=2):
    """n rows of `entries` (odd) entries each: a ring of neighbours."""
    i = np.arange(n)[:, None]
    off = np.arange(-(entries // 2), entries // 2 + 1)
    col = np.sort((i + off) % n, axis=1).astype(np.int32)
    u = np.random.default_rng(seed)
    val = np.full(col.shape, -1.0)
    val[col == i] = entries + 0.5
    dia = (np.nonzero(col.ravel() == np.repeat(np.arange(n), entries))[0]).astype(np.int32)
    return ((np.arange(n + 1) * entries).astype(np.int32), col.ravel(), dia, val.ravel(),
            u.uniform(-1, 1, n))


@pytest.mark.parametrize("entries,vectors", [(3, 8), (19, 8), (21, 7), (151, 7)])
@pytest.mark.parametrize("n", [400, 6007])
def test_direction(oracle, n, entries, vectors):
    import torch
    from tflows_amd import solvers as S
    if not torch.cuda.is_available():
        pytest.fail("no GPU visible")
    row, col, dia, val, b = band(n, entries)
    print(f"direction n={n} entries={entries}", flush=True)
    A = S.Matrix(row, col, dia, val)
    before = A.info()["device_bytes"]
    tol = 1e-10 * float(np.linalg.norm(b))
    x, r = torch.zeros(n, dtype=torch.float64, device="cuda"), torch.from_numpy(b).cuda()
    niter, _, fin = S.solve("cg", A, x, r, 1, 1000, tol)
    assert A.info()["device_bytes"] - before == 8 * n * vectors
    ref = oracle.solve("cg", row, col, dia, val, b, prec=1, niter=1000, tol=tol)
    assert abs(niter - ref["niter"]) <= max(1, ref["niter"] // 20) and fin < tol
    assert rel_l2(x.cpu().numpy(), ref["x"]) <= 1e-8
