"""Structures whose blocks are nearly empty (small systems side by side, chains)
have block sweeps only as long as staging their blocks costs less than the
levels do."""
import numpy as np
import pytest

from test_gpu_blocks import nine_point
from tflows_amd import mesh


def side_by_side(row, col, dia, k):
    n, z = len(dia), len(col)
    at = np.arange(k)[:, None]
    return (np.concatenate(([0], (row[1:] + at * z).ravel())).astype(np.int32),
            (col + at * n).ravel().astype(np.int32), (dia + at * z).ravel().astype(np.int32))


def box(*d):
    c = mesh.make_case(nx=d[0], ny=d[1], nz=d[2])
    return c.row, c.col, c.dia


# us per sweep on MI355X, levels / blocks, beside each
@pytest.mark.parametrize("system,count,blocks", [
    (lambda: box(9, 9, 9), 274, True),                # 37 / 19
    (lambda: box(9, 9, 9), 1371, False),              # 42 / 73
    (lambda: box(1, 1, 32), 625, True),               # 36 / 15
    (lambda: box(1, 1, 32), 6250, False),             # 43 / 125
    (lambda: box(12, 12, 12), 115, True),             # 49 / 15
    (lambda: box(17, 17, 3), 1153, False),            # 55 / 71
    (lambda: nine_point(12, 12)[:3], 347, True),      # 50 / 29
    (lambda: nine_point(12, 12)[:3], 1388, False),    # 51 / 103
])
def test_nearly_empty_blocks(system, count, blocks):
    row, col, dia = side_by_side(*system(), count)
    assert (mesh.layout_blocks(row, col, dia) is not None) == blocks


def test_full_blocks_stay():
    c = mesh.make_case(nx=80)
    assert mesh.layout_blocks(c.row, c.col, c.dia) is not None
