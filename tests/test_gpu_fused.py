"""CG and CGS iterations whose sums end in the summing kernel and whose
direction is formed in the product, at the sizes where each starts or ends:
five iterations against the oracle.  Sums of n products in another order differ
by at most n eps = 3e-11 relative (n = 2^17); few rounding errors are as bad."""
import numpy as np
import pytest

from tflows_amd import mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1, 1, 1), (5, 13, 1), (16, 16, 4), (41, 5, 5), (32, 32, 32),
                                  (32, 32, 33), (32, 32, 64), (32, 32, 65), (32, 64, 64),
                                  (32, 64, 65)])
@pytest.mark.parametrize("method,prec", [("cg", 2), ("cg", 1), ("cg", 0), ("cgs", 2)])
def test_iterations(oracle, dims, method, prec):
    import torch
    from tflows_amd import solvers
    c = mesh.make_case(kind=mesh.MOMENTUM, nx=dims[0], ny=dims[1], nz=dims[2], beta=1.0,
                       pin_first=False, rhs_zero_mean=False)
    print(f"fused {dims} {method} prec {prec}", flush=True)
    A = solvers.Matrix(c.row, c.col, c.dia, c.val)
    tol = 1e-13 * float(np.linalg.norm(c.b))
    ref = oracle.solve(method, c.row, c.col, c.dia, c.val, c.b, prec=prec, niter=5, tol=tol)
    for _ in range(2):   # the second solve starts from the first one's buffers
        x = torch.zeros(c.n, dtype=torch.float64, device="cuda")
        r = torch.from_numpy(c.b.copy()).cuda()
        niter, ini, fin = solvers.solve(method, A, x, r, prec, 5, tol)
        assert niter == ref["niter"]
        assert np.linalg.norm(x.cpu().numpy() - ref["x"]) <= 3e-11 * np.linalg.norm(ref["x"])
