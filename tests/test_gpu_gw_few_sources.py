"""GPU test of lem_gw_mfma with few sources that are not padding: the products of a G
factor and a weight are as accurate as float32 arithmetic makes them, one by one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# k_gw_mfma with one and with eight wavefronts a tile, k_gw_tile
@pytest.mark.parametrize("S,K,F", [(32, 96, 1), (1024, 2720, 1), (64, 16416, 3)])
def test_one_source_as_accurate_as_float32(native, S, K, F):
    rng = np.random.default_rng(S)
    src = rng.uniform(-0.5, 0.5, (S, 3)).astype(np.float32)
    snk = (rng.normal(size=(K, 3)) * 3 + [0, 0, 12]).astype(np.float32)
    n = rng.normal(size=(K, 3))
    n = (n / np.linalg.norm(n, axis=1, keepdims=True)).astype(np.float32)
    kf, pol = np.linspace(60.0, 90.0, F), np.array([0.6, 0.0, 0.8], np.float32)
    w = (rng.normal(size=64) + 1j * rng.normal(size=64)).astype(np.complex64)
    for s in (0, S - 11):
        W = np.zeros((F, S, 64), np.complex64)
        W[:, s] = 1
        G = native.gw_mfma(src, pol, snk, n, kf, W).cpu().numpy()
        assert np.array_equal(G, np.broadcast_to(G[..., :1], G.shape))  # G 1 = G, exactly
        W[:, s] = w
        got = native.gw_mfma(src, pol, snk, n, kf, W).cpu().numpy()
        g, x = G.astype(np.complex128), w.astype(np.complex128)
        err = got - g * x
        for e, terms, sign in (
                (err.real, np.abs(g.real * x.real) + np.abs(g.imag * x.imag), (g * x).real),
                (err.imag, np.abs(g.real * x.imag) + np.abs(g.imag * x.real), (g * x).imag)):
            e = e / terms * 2.0 ** 24
            # float32 arithmetic rounds twice, each time by at most half a unit in the
            # last place, 1 here, and evenly: sqrt(2 / 3) in the mean square, none in
            # the mean.  The means are over thousands of values of g for 64 of w.
            assert np.sqrt(np.mean(e * e)) <= np.sqrt(2 / 3)
            assert abs(np.mean(e * np.sign(sign))) <= 0.1
            # and one by one: both roundings, and 2^-24 of each product left out
            assert np.abs(e).max() <= 4


def test_attenuation_is_not_rounded_before_the_path(native):
    """exp(-alpha r) over 900 to 1,100 m at alpha = 0.05: the float32 nearest to 0.05 is
    1.5e-8 of it away, 7.5e-7 of the field at 1 km.  What is left on average are the
    constants of the factor (front, wavenumber), each off by at most 2^-24 = 6e-8, and
    1/r to a unit in the last place, 1.2e-7; the exponent's own rounding, 50 2^-24 / sqrt 3
    at a time, averages to 3e-8 over 4,096 sinks."""
    rng = np.random.default_rng(3)
    K, S, alpha, kf = 4096, 32, 0.05, np.array([41.9])
    src = np.zeros((S, 3), np.float32)
    u = rng.normal(size=(K, 3))
    u[:, 2] = 0.0
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    snk = (u * rng.uniform(900.0, 1100.0, (K, 1))).astype(np.float32)
    W = np.zeros((1, S, 64), np.complex64)
    W[:, 3] = 1
    got = native.gw_mfma(src, np.array([0, 0, 1], np.float32), snk, u.astype(np.float32), kf, W,
                         alpha=alpha).cpu().numpy()[0, 2, :, 0]
    d = snk.astype(np.float64)
    r = np.linalg.norm(d, axis=1)
    want = np.exp(-alpha * r) / r / (2 * np.pi) * np.abs(alpha + 1j * kf[0] + 1 / r) * \
        np.einsum("kc,kc->k", d / r[:, None], u.astype(np.float32).astype(np.float64))
    assert abs(np.mean(np.abs(got) / want - 1)) <= 3e-7
