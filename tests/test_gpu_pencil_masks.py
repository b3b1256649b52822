"""GPU tests of the grid walks of clustered points (pencils and beams) against the dense
kernel where pairs of one row are left out, in grids whose macro blocks are 4 x 4 x 4
cells and larger ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 768  # N x N rays are enough for the beams and pencils


def _terrain(rng, n):
    h = rng.normal(size=(n + 1, n + 1))
    i, j = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")

    def v(a, b):
        return np.stack([a, b, h[a, b]], -1).reshape(-1, 3)

    p00, p10, p01, p11 = v(i, j), v(i + 1, j), v(i, j + 1), v(i + 1, j + 1)
    return np.concatenate([np.concatenate([p00, p10, p11], 1),
                           np.concatenate([p00, p11, p01], 1)]).astype(np.float32)


@pytest.fixture(scope="module", params=[40, 300])
def scene(request, native):
    """Four clusters of 192 points above and below a terrain, each a fraction of a cell
    wide: most words of 64 lie in one of them."""
    n = request.param
    rng = np.random.default_rng(n)
    tris = _terrain(rng, n)
    g = native.Grid(tris)
    # pencils: 4 x 4 x 4 cells are one macro block, or several sub-blocks of one
    assert (g.info.mshift == 2) == (n == 40) and g.info.mshift <= 4
    width = 0.2 * min(g.info.cell)

    def clusters(z):
        c = np.c_[rng.uniform(0.2 * n, 0.8 * n, (4, 2)), z]
        return np.repeat(c, 192, 0) + rng.uniform(-width, width, (N, 3))

    # two clusters' own pairs pass through the terrain, two do not
    src, snk = clusters([5.0, 5.0, 5.0, -5.0]), clusters([-5.0, -5.0, 5.0, -5.0])
    return tris, g, src.astype(np.float32), snk.astype(np.float32)


def _mask(bits, n):
    return np.unpackbits(bits.cpu().numpy().view(np.uint8), axis=1, bitorder="little")[:, :n]


@pytest.mark.parametrize("from_sink", [False, True])
@pytest.mark.parametrize("sink_major", [False, True])
@pytest.mark.parametrize("skip_self", [False, True])
def test_pencils_leave_out_pairs_of_one_row(native, scene, skip_self, sink_major, from_sink):
    tris, g, src, snk = scene
    want = _mask(native.visibility_dense(src, snk, tris, skip_self=skip_self)[0], N)
    got = _mask(g.visibility(src, snk, skip_self=skip_self, sink_major=sink_major,
                             from_sink=from_sink)[0], N)
    assert np.array_equal(want, got.T if sink_major else got)
    # half of the pairs' own rays would be blocked, in words that are blocked as a whole
    assert np.diag(want).sum() == 0 if skip_self else np.diag(want).mean() > 0.4
    assert 0.2 < want.mean() < 0.9


@pytest.mark.parametrize("sink_major", [False, True])
def test_closest_hits_leave_out_pairs_of_one_row(native, scene, sink_major):
    tris, g, src, snk = scene
    want, wd = native.visibility_dense(src, snk, tris, skip_self=True, any_hit=False,
                                       want_dist=True)
    got, gd = g.visibility(src, snk, skip_self=True, any_hit=False, want_dist=True,
                           sink_major=sink_major)
    want, got = _mask(want, N), _mask(got, N)
    wd, gd = wd.cpu().numpy(), gd.cpu().numpy()
    assert np.array_equal(want, got.T if sink_major else got)
    assert np.array_equal(wd, gd.T if sink_major else gd)
    assert np.diag(want).sum() == 0


@pytest.mark.parametrize("sink_major", [False, True])
@pytest.mark.parametrize("narrow", [0.7, 0.8, 1.0])
def test_wide_words_among_pencils(native, scene, narrow, sink_major):
    """Points of one cluster and points all over the scene, on either side of the share
    from which pencils are cast, and points along a line."""
    tris, g, src, snk = scene
    rng = np.random.default_rng(5)
    side = tris.reshape(-1, 3).max()
    n = int(narrow * 4096)
    lanes = np.empty((4096, 3), np.float32)
    lanes[:n] = rng.uniform(0, 0.2 * min(g.info.cell), (n, 3)) + [0.5 * side, 0.4 * side, 5.0]
    lanes[n:] = rng.uniform([0, 0, -6], [side, side, 6], (4096 - n, 3))
    line = np.linspace(0.1, 0.9, 4096)[:, None] * np.array([side, 0, 0]) + [0, 0.3 * side, 5.0]
    for points in (lanes, line.astype(np.float32)):
        a, b = (points, snk) if sink_major else (snk, points)
        want = _mask(native.visibility_dense(a, b, tris)[0], len(b))
        for from_sink in (False, True):
            got = _mask(g.visibility(a, b, sink_major=sink_major, from_sink=from_sink)[0], len(points))
            assert np.array_equal(want, got.T if sink_major else got)
