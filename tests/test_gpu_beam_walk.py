"""GPU tests of the beam walk of the persistent grid traversal against the dense
kernel, which tests every triangle: lanes on either side, closest and any hit, words
cut short, narrow and wide words, rays along grid planes and zero-length rays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _terrain(rng, n=40):
    h = rng.normal(size=(n + 1, n + 1))
    i, j = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")

    def v(a, b):
        return np.stack([a, b, h[a, b]], -1).reshape(-1, 3)

    p00, p10, p01, p11 = v(i, j), v(i + 1, j), v(i, j + 1), v(i + 1, j + 1)
    return np.concatenate([np.concatenate([p00, p10, p11], 1),
                           np.concatenate([p00, p11, p01], 1)]).astype(np.float32)


def _points(rng, kind, n):
    if kind == "grid":      # rows above the terrain; many rays along grid planes
        side = int(np.ceil(np.sqrt(n)))
        x, y = np.meshgrid(np.linspace(1, 39, side), np.linspace(1, 39, side), indexing="ij")
        p = np.stack([x.ravel(), y.ravel(), np.full(side * side, 4.0)], 1)[:n]
    elif kind == "clusters":
        c = rng.uniform([0, 0, -1], [40, 40, 6], (n // 64 + 1, 3))
        p = (np.repeat(c, 64, 0) + rng.normal(size=(64 * (n // 64 + 1), 3)) * 0.05)[:n]
    elif kind == "pencil":  # all within a fraction of a cell
        p = rng.normal(size=(n, 3)) * 0.02 + [20.0, 20.0, 4.0]
        p[:n // 2, 2] = 4.0
    else:                   # far origins
        p = rng.normal(size=(n, 3)) * 5 + [2000.0, -1500.0, 900.0]
    return p.astype(np.float32)


@pytest.mark.parametrize("kind,n", [("grid", 8191), ("grid", 65536), ("clusters", 20000),
                                    ("far", 12345), ("pencil", 8000)])
@pytest.mark.parametrize("sink_major", [True, False])
def test_beams_equal_the_dense_masks(native, kind, n, sink_major):
    rng = np.random.default_rng(n)
    tris = _terrain(rng)
    lanes = _points(rng, kind, n)
    outer = rng.uniform([0, 0, -0.5], [40, 40, 5], (530, 3)).astype(np.float32)
    outer[:20, 2] = 4.0          # along the grid of points
    outer[20:24] = lanes[:4]     # zero-length rays
    assert lanes.shape[0] * outer.shape[0] >= 1 << 22
    src, snk = (lanes, outer) if sink_major else (outer, lanes)
    g = native.Grid(tris)
    for any_hit in (False, True):
        want, dist = native.visibility_dense(src, snk, tris, any_hit=any_hit,
                                             want_dist=not any_hit)
        got, gd = g.visibility(src, snk, any_hit=any_hit, want_dist=not any_hit,
                               sink_major=sink_major)
        # rows of either are words of 64 bits along the lanes' side
        a = np.unpackbits(want.cpu().numpy().view(np.uint8), axis=1, bitorder="little")
        b = np.unpackbits(got.cpu().numpy().view(np.uint8), axis=1, bitorder="little")
        a, b = a[:, :len(snk)], b[:, :len(lanes)]
        assert np.array_equal(a.T if sink_major else a, b)
        assert 0.01 < a.mean() < 0.99
        if not any_hit:
            d = dist.T if sink_major else dist
            assert np.array_equal(d.cpu().numpy(), gd.cpu().numpy(), equal_nan=True)


def test_beams_skip_self(native):
    rng = np.random.default_rng(1)
    tris = _terrain(rng)
    p = _points(rng, "grid", 2100)
    g = native.Grid(tris)
    want, _ = native.visibility_dense(p, p, tris, skip_self=True)
    got, _ = g.visibility(p, p, skip_self=True)
    assert np.array_equal(want.cpu().numpy(), got.cpu().numpy())
