"""The server's device bytes stay within the budget whatever preconditioners a
resident case's requests ask for, one after another."""
import numpy as np
import pytest

from tflows_amd import mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [(0, 1, 2), (2, 0, 1), (1, 2, 0)])
def test_preconditioners_in_turn(order):
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no GPU visible")
    from tflows_amd import solvers as S
    cs = [mesh.make_case(kind=mesh.MOMENTUM, nx=k, beta=2.0, jitter=0.1, permute=True,
                         pin_first=False, rhs_zero_mean=False) for k in (24, 30)]

    def ask(srv, cid, c, prec):
        h = srv.submit(cid, "cg", prec, c.b, 1e-6 * float(np.linalg.norm(c.b)), 500)
        assert srv.wait(h)["status"] >= 0   # converged or not: its memory counts

    srv = S.Server(1 << 30, workers=1)
    ids = [srv.add_case(c.row, c.col, c.dia, c.val) for c in cs]
    for cid, c in zip(ids, cs):
        ask(srv, cid, c, order[0])
    held = srv.stats()["hbm_in_use"]
    for prec in order[1:]:
        for cid, c in zip(ids, cs):
            ask(srv, cid, c, prec)
            assert srv.stats()["hbm_in_use"] == held
    srv.close()
