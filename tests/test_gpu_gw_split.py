"""GPU tests of the two kernels behind lem_gw_mfma (three-part bfloat16 products): the
edges of their tiles and source splits against float64, scaled weights, and weights
that are not finite."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# one workgroup of k_gw_tile (half of its sinks missing; whole; one and a half), then
# k_gw_mfma with the sources split over 2, 4 and 8 wavefronts, evenly and not, then
# k_gw_tile again with several frequencies
SHAPES = [(32, 32, 1), (64, 64, 2), (32, 96, 1), (128, 32, 1), (224, 96, 2), (992, 64, 1),
          (1024, 2720, 1), (64, 16416, 3)]


def _case(S, K, F, seed=1):
    rng = np.random.default_rng(seed)
    src = rng.uniform(-0.5, 0.5, (S, 3)).astype(np.float32)
    snk = (rng.normal(size=(K, 3)) * 3 + [0, 0, 12]).astype(np.float32)
    n = rng.normal(size=(K, 3))
    n = (n / np.linalg.norm(n, axis=1, keepdims=True)).astype(np.float32)
    W = (rng.normal(size=(F, S, 64)) + 1j * rng.normal(size=(F, S, 64))).astype(np.complex64)
    pol = np.array([0.6, 0.0, 0.8], np.float32)
    return src, pol, snk, n, np.linspace(60.0, 90.0, F), W


def _exact(src, pol, snk, n, kf, W, alpha, sinks):
    """float64 E and the sums of |G| |W| that bound its rounding errors."""
    d = snk[sinks].astype(np.float64)[:, None] - src.astype(np.float64)[None]
    r = np.linalg.norm(d, axis=2)
    u = d / r[..., None]
    e = pol.astype(np.float64)
    p = e - u * (u @ e)[..., None]
    cs = np.einsum("ksc,kc->ks", u, n[sinks].astype(np.float64))
    E, bound = [], []
    for f, k in enumerate(kf):
        F_ = np.exp(-(alpha + 1j * k) * r) / r * (-1 / (2 * np.pi)) * (-(alpha + 1j * k) - 1 / r)
        G = ((F_ * cs)[..., None] * p).transpose(2, 0, 1)
        E.append(G @ W[f].astype(np.complex128))
        bound.append(np.abs(G) @ np.abs(W[f]).astype(np.float64))
    return np.stack(E), np.stack(bound)


@pytest.mark.parametrize("alpha", [0.0, 0.05])
@pytest.mark.parametrize("S,K,F", SHAPES)
def test_gw_split_against_float64(native, S, K, F, alpha):
    src, pol, snk, n, kf, W = _case(S, K, F)
    got = native.gw_mfma(src, pol, snk, n, kf, W, alpha=alpha).cpu().numpy()
    sinks = np.unique(np.r_[0:min(K, 40), max(0, K - 70):K])
    ref, bound = _exact(src, pol, snk, n, kf, W, alpha, sinks)
    # G is a chain of about 16 float32 operations, each 2^-24 of a value no larger than
    # twice the factor (p cancels); the sums add less than 24 of the terms' sum in all
    # (16 sources a step, S / 16 steps, every rounding of random sign)
    assert np.all(np.abs(got[:, :, sinks] - ref) <= 64 * 2.0 ** -24 * bound + 1e-12)
    assert np.linalg.norm(got[:, :, sinks] - ref) <= 2e-6 * np.linalg.norm(ref)


@pytest.mark.parametrize("S,K", [(64, 96), (992, 64)])
def test_gw_split_scales_with_the_weights(native, S, K):
    """Powers of two up to the ends of float32 leave every part's bits alone."""
    src, pol, snk, n, kf, W = _case(S, K, 1)
    one = native.gw_mfma(src, pol, snk, n, kf, W).cpu().numpy()
    for e in (-80, 100):
        got = native.gw_mfma(src, pol, snk, n, kf, W * np.float32(2.0 ** e)).cpu().numpy()
        assert np.array_equal(got, one * np.float32(2.0 ** e))


@pytest.mark.parametrize("S,K", [(64, 96), (992, 64)])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_gw_split_weights_that_are_not_finite(native, S, K, bad):
    src, pol, snk, n, kf, W = _case(S, K, 2)
    one = native.gw_mfma(src, pol, snk, n, kf, W).cpu().numpy()
    W2 = W.copy()
    W2[1, S - 3, 37] = bad
    got = native.gw_mfma(src, pol, snk, n, kf, W2).cpu().numpy()
    hit = np.zeros(one.shape, bool)
    hit[1, :, :, 37] = True
    assert not np.isfinite(got[hit]).any()
    if not np.isnan(bad):  # float32 arithmetic: (gr + i gi) (inf + 0i), no NaN but for 0 * inf
        d, _ = _exact(src[S - 3:S - 2], pol, snk, n, kf[1:], np.ones((1, 1, 1), np.complex64),
                      0.0, np.arange(K))
        assert np.array_equal(np.sign(got[1, :, :, 37].real), np.sign(bad * d[0, :, :, 0].real))
    # the rest of the tiles it touches is done with the FP32 instructions
    assert np.linalg.norm(got[~hit] - one[~hit]) <= 2e-6 * np.linalg.norm(one[~hit])
