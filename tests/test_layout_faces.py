"""The cells' face lists of the device face loops (tfs_layout_faces): every
cell's entries are its faces, ascending, with its side; the cells are taken in
the face list's order where their own numbering scatters, else in the caller's."""
import numpy as np
import pytest

from tflows_amd import mesh


def expected(n, faces, base):
    c1, c2 = faces[0::2] - base, faces[1::2] - base
    s = np.arange(len(c1))
    cell = np.concatenate((c1, c2[c2 >= 0]))
    entry = np.concatenate((2 * s, 2 * s[c2 >= 0] + 1))
    k = np.lexsort((entry // 2 * 2 + entry % 2, cell))
    return np.concatenate(([0], np.cumsum(np.bincount(cell, minlength=n)))), entry[k]


def check(n, faces, base, reorder_from=2):
    reordered, order, first, entry = mesh.layout_faces(n, faces, base, reorder_from)
    want_first, want_entry = expected(n, faces, base)
    assert np.array_equal(first, want_first) and np.array_equal(entry, want_entry)
    assert np.array_equal(np.sort(order), np.arange(n))
    assert reordered or np.array_equal(order, np.arange(n))
    return reordered


@pytest.mark.parametrize("dims", [(1, 1, 1), (4, 4, 4), (5, 13, 1), (30, 31, 17)])
@pytest.mark.parametrize("permute", [False, True])
def test_box(dims, permute):
    c = mesh.make_case(nx=dims[0], ny=dims[1], nz=dims[2], permute=permute, with_faces=True)
    reordered = check(c.n, c.faces, 1)
    assert reordered == (permute and c.n > 10000)
    assert not check(c.n, c.faces, 1, c.n + 1)


@pytest.mark.parametrize("base", [0, 1])
@pytest.mark.parametrize("spokes", [31, 32, 33, 64, 200])
def test_tails(base, spokes):
    """A cell of many faces beside ordinary ones, and cells of none."""
    n = spokes + 70
    f = [(3, 4 + k) if k % 2 else (4 + k, 3) for k in range(spokes - 1)] + [(3, -1), (n - 1, 0)]
    check(n, (np.array(f) + base).reshape(-1).astype(np.int32), base)


def test_random_faces():
    """No order to be had from the faces: the caller's stays."""
    u = np.random.default_rng(1)
    f = u.integers(1, 5001, (20000, 2))
    f[f[:, 0] == f[:, 1], 1] = 0
    assert not check(5000, f.reshape(-1).astype(np.int32), 1)
