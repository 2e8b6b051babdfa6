"""Cells of more faces than a slice has slots for, in a mesh whose cells the face
lists take in another order than the caller's: the tails go by position."""
import numpy as np
import pytest

from test_layout_faces import check
from tflows_amd import mesh


def with_hub(dims, extra, seed=1):
    """A randomly numbered box one of whose cells has `extra` more faces."""
    c = mesh.make_case(nx=dims[0], ny=dims[1], nz=dims[2], permute=True, with_faces=True)
    f = c.faces.reshape(-1, 2)
    u = np.random.default_rng(seed)
    hub = int(u.integers(1, c.n + 1))
    near = np.concatenate((f[f[:, 0] == hub, 1], f[f[:, 1] == hub, 0], [hub]))
    to = np.setdiff1d(u.permutation(c.n)[:extra + len(near)] + 1, near)[:extra]
    mine = np.stack((np.full(extra, hub), to), axis=1)
    mine[::2] = mine[::2, ::-1]          # second as well as first in its faces
    at = np.sort(u.integers(0, len(f) + 1, extra))
    return c.n, np.insert(f, at, mine, axis=0).astype(np.int32).ravel(), hub


@pytest.mark.parametrize("extra", [20, 27, 40, 300])
def test_reordered_tails(extra):
    n, faces, hub = with_hub((30, 31, 17), extra)
    assert check(n, faces, 1)                      # reordered, and every list as expected
    _, order, first, _ = mesh.layout_faces(n, faces, 1, 2)
    assert first[hub] - first[hub - 1] >= extra and order[hub - 1] != hub - 1
