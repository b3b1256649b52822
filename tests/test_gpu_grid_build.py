"""GPU tests of the grid build against numpy: reference lists of every length the sorts
treat differently, triangles in mesh order and shuffled, large and degenerate ones,
and the macro blocks' boxes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _tris(kind, T, rng):
    if kind == "mesh":        # neighbours share cells
        n = int(np.ceil(np.sqrt(T / 2)))
        i, j = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
        h = rng.normal(size=(n + 1, n + 1))

        def v(a, b):
            return np.stack([a, b, h[a, b]], -1).reshape(-1, 3)

        t = np.stack([np.concatenate([v(i, j), v(i + 1, j), v(i + 1, j + 1)], 1),
                      np.concatenate([v(i, j), v(i + 1, j + 1), v(i, j + 1)], 1)], 1)
        t = t.reshape(-1, 9)[:T]
    else:
        c = rng.uniform(-1, 1, (T, 1, 3))
        size = {"small": 0.02, "large": 0.7, "heap": 1e-4}[kind]
        if kind == "heap":    # lists far longer than 32
            c = np.round(c)
        t = (c + rng.uniform(-size, size, (T, 3, 3))).reshape(T, 9)
        t[::17, 3:6] = t[::17, 0:3]
    return t.astype(np.float32)


@pytest.mark.parametrize("kind", ["mesh", "small", "large", "heap"])
@pytest.mark.parametrize("T,cells", [(1, 2.0), (63, 2.0), (65, 0.2), (3000, 0.05), (5000, 2.0),
                                     (20001, 8.0)])
@pytest.mark.parametrize("shuffled", [False, True])
def test_grid_build(native, kind, T, cells, shuffled):
    rng = np.random.default_rng(T)
    tris = _tris(kind, T, rng)
    if shuffled:
        tris = tris[rng.permutation(T)]
    g = native.Grid(tris, cells_per_tri=cells)
    f = np.float32
    lo = np.array([g.info.lo[a] for a in range(3)], f)
    cell = np.array([g.info.cell[a] for a in range(3)], f)
    n = np.array([g.info.n[a] for a in range(3)])
    v = tris.reshape(T, 3, 3)
    eps = f(g.info.eps)
    a = np.clip(np.floor((v.min(1) - eps - lo) * (f(1) / cell)).astype(int), 0, n - 1)
    b = np.clip(np.floor((v.max(1) + eps - lo) * (f(1) / cell)).astype(int), 0, n - 1)
    cells_of, ids_of = [], []
    for t in range(T):
        z, y, x = np.meshgrid(*[np.arange(a[t, i], b[t, i] + 1) for i in (2, 1, 0)],
                              indexing="ij")
        cells_of.append(((z * n[1] + y) * n[0] + x).ravel())
        ids_of.append(np.full(x.size, t))
    c, ids = np.concatenate(cells_of), np.concatenate(ids_of)
    order = np.lexsort((ids, c))
    nc = int(n.prod())
    start = np.r_[0, np.cumsum(np.bincount(c, minlength=nc))]
    assert g.info.ncells == nc and g.info.nrefs == len(c)
    assert np.array_equal(g.cell_start.cpu().numpy(), start)
    assert np.array_equal(g.tri_ids.cpu().numpy()[:len(c)], ids[order])
    box = g.cell_box.cpu().numpy()[:8 * (nc + g.info.nmacro)].reshape(-1, 2, 4)[:, :, :3]
    B = 1 << g.info.mshift
    m = -(-n // B)
    z, y, x = np.unravel_index(np.arange(nc), n[::-1])
    block = ((z // B) * m[1] + y // B) * m[0] + x // B
    want = np.empty((g.info.nmacro, 2, 3), f)
    want[:, 0], want[:, 1] = np.inf, -np.inf
    np.minimum.at(want[:, 0], block, box[:nc, 0])
    np.maximum.at(want[:, 1], block, box[:nc, 1])
    assert np.array_equal(box[nc:], want)
