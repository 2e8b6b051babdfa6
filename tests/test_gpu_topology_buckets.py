"""The topology by buckets of cells (meshes of 2^15 cells and more) bitwise
against the host builder: at the size where it starts, with a last bucket that
is not full, rows of every sorting width, repeated pairs and faces of a cell
with itself, without positions, and where a bucket does not fit."""
import numpy as np
import pytest

from tflows_amd import mesh

pytestmark = pytest.mark.gpu


def box(permute, *d):
    c = mesh.make_case(nx=d[0], ny=d[1], nz=d[2], permute=permute, with_faces=True)
    return c.n, c.faces


def uneven(n, nf, crowd=0):
    """Random pairs among clustered cells (rows of 1 to about 40), repeated pairs,
    faces of a cell with itself, boundary faces; `crowd` faces among 1000 cells."""
    u = np.random.default_rng(n)
    c1 = (n * u.random(nf) ** 2).astype(np.int64) + 1
    c2 = np.clip(c1 + u.integers(-300, 300, nf), -50, n)
    c2[c2 == 0] = -1
    c2[::100] = c1[::100]
    c1[1::7], c2[1::7] = c1[0::7][:len(c1[1::7])], c2[0::7][:len(c2[1::7])]
    c1[:crowd], c2[:crowd] = u.integers(1, 1001, crowd), u.integers(1, 1001, crowd)
    return n, np.stack((c1, c2), 1).reshape(-1).astype(np.int32)


MESHES = {
    "32^3": lambda: box(False, 32, 32, 32), "32^3 permuted": lambda: box(True, 32, 32, 32),
    "odd": lambda: box(False, 61, 43, 37), "odd permuted": lambda: box(True, 61, 43, 37),
    "thin": lambda: box(True, 1, 257, 151), "uneven": lambda: uneven(50001, 150000),
    "dense": lambda: uneven(40000, 700000), "crowd": lambda: uneven(40000, 120000, 12000),
}


@pytest.mark.parametrize("name", MESHES)
@pytest.mark.parametrize("base", [0, 1])
def test_topology(name, base):
    import torch
    from tflows_amd import solvers
    n, faces = MESHES[name]()
    print(f"topology {name} n={n} nf={faces.size // 2} base={base}", flush=True)
    want = mesh.topology(n, faces, base=base, with_pos=True)
    f = torch.from_numpy(faces).cuda()
    got = solvers.topology_device(n, f, base=base)
    for what, w, g in zip(("row", "col", "dia", "pos"), want, got):
        assert np.array_equal(g.cpu().numpy(), w), what
    got = solvers.topology_device(n, f, base=base, with_pos=False)
    for what, w, g in zip(("row", "col", "dia"), want, got):
        assert np.array_equal(g.cpu().numpy(), w), what
    f[2 * (faces.size // 4)] = n + 1
    with pytest.raises(solvers.SolverError):
        solvers.topology_device(n, f, base=base)
