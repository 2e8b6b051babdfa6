"""Blocks of the FP64 sweeps (tfs_layout_blocks): every row's earlier
neighbours sit in earlier blocks or in earlier steps of its own block, in the
order the kernel walks; and the structures that have no blocks."""
import numpy as np
import pytest

from tflows_amd import mesh

BOXES = [(9, 9, 9), (12, 12, 12), (61, 23, 40), (2, 3, 60), (1, 1, 100), (30, 1, 40), (17, 64, 9)]


@pytest.mark.parametrize("dims", BOXES)
def test_order_and_limits(dims):
    c = mesh.make_case(nx=dims[0], ny=dims[1], nz=dims[2])
    nblk, order, block, step = mesh.layout_blocks(c.row, c.col, c.dia)
    assert np.array_equal(np.sort(order), np.arange(c.n))
    assert np.all(np.diff(block[order]) >= 0) and block.max() == nblk - 1
    row_of = np.repeat(np.arange(c.n), np.diff(c.row))
    low = c.col < row_of
    i, j = row_of[low], c.col[low]
    before = (block[j] < block[i]) | ((block[j] == block[i]) & (step[j] < step[i]))
    assert before.all()
    _, rows = np.unique(block, return_counts=True)
    _, lanes = np.unique(block.astype(np.int64) * 64 + step, return_counts=True)
    assert rows.max() <= 512 and lanes.max() <= 64 and step.max() < 63


def test_box_blocks_are_bricks():
    """On a lexicographic box the blocks are 8^3 bricks whatever the sides' order."""
    for dims in ((24, 16, 40), (16, 24, 40), (40, 16, 24)):
        c = mesh.make_case(nx=dims[0], ny=dims[1], nz=dims[2])
        nblk, _, block, _ = mesh.layout_blocks(c.row, c.col, c.dia)
        x, y, z = np.arange(c.n) % dims[0], np.arange(c.n) // dims[0] % dims[1], \
            np.arange(c.n) // (dims[0] * dims[1])
        brick = (x // 8) + 100 * ((y // 8) + 100 * (z // 8))
        assert nblk == dims[0] * dims[1] * dims[2] // 512
        assert len(np.unique(np.stack((block, brick)), axis=1)[0]) == nblk


def test_structures_without_blocks():
    c = mesh.make_case(nx=14, permute=True)
    assert mesh.layout_blocks(c.row, c.col, c.dia) is None       # too shallow
    c = mesh.make_case(nx=16)
    keep = np.ones(c.nnz, bool)
    keep[c.row[100]] = False                                     # one pair loses its mirror
    row = np.concatenate(([0], np.cumsum([keep[c.row[i]:c.row[i + 1]].sum()
                                          for i in range(c.n)]))).astype(np.int32)
    dia = (np.cumsum(keep)[c.dia] - 1).astype(np.int32)
    assert mesh.layout_blocks(row, c.col[keep], dia) is None     # not symmetric
    assert mesh.layout_blocks(c.row, c.col, c.dia) is not None
