"""A batch holds no copy of the caller's rows: only products of a matrix's own
vectors read one, and a batch has none."""
import numpy as np
import pytest

from tflows_amd import mesh

pytestmark = pytest.mark.gpu


def test_no_callers_rows():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no GPU visible")
    from tflows_amd import solvers as S
    small = mesh.make_case(nx=8)
    S.Matrix(small.row, small.col, small.dia, small.val).close()   # the library's own arrays
    c = mesh.make_case(nx=80)

    def held(make):
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        obj = make()
        took = free - torch.cuda.mem_get_info()[0]
        obj.close()
        return took

    matrix = held(lambda: S.Matrix(c.row, c.col, c.dia, c.val))
    batch = held(lambda: S.Batch([(c.row, c.col, c.dia, c.val)]))
    rows = 4 * (c.nnz + c.n)
    print(f"matrix {matrix} batch {batch} rows {rows}", flush=True)
    assert batch <= matrix - rows + (4 << 20)   # a batch's own arrays are small
