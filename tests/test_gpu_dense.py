"""lem_visibility_dense (shared-origin tests, rays sorted by direction) against
lem_raycast_pairs, which runs the predicate on every triangle: masks and
distances equal, at the edges of the workgroups and triangle tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _scene(K, T, seed):
    rng = np.random.default_rng(seed)
    src = rng.uniform(-0.5, 0.5, (3, 3)).astype(np.float32)
    snk = rng.uniform(-4, 4, (K, 3)).astype(np.float32)
    snk[0] = src[1]                        # a zero-length ray
    snk[K // 2] = src[0] + [0, 0, 2]       # a ray along an axis
    v = rng.uniform(-3, 3, (T, 1, 3)) + rng.uniform(-0.6, 0.6, (T, 3, 3))
    tris = v.reshape(T, 9).astype(np.float32)
    if T >= 8:
        tris[1] = tris[0]                                  # the same triangle twice (a tie)
        tris[2, 6:] = tris[2, 3:6]                         # degenerate
        tris[3] = np.concatenate([src[0], src[0] + [1, 0, 0], src[0] + [0, 1, 0]])  # through an origin
        tris[4] *= np.float32(1e20)                        # overflows the products
        tris[5, 0] = np.nan
        tris[6, 2::3] = src[0, 2]                          # an origin in its plane
    return src, snk, tris


@pytest.mark.parametrize("K,T", [(1, 1), (63, 7), (64, 127), (65, 128), (255, 256), (257, 257),
                                 (700, 640), (4095, 300), (4096, 300), (4609, 513)])
@pytest.mark.parametrize("mode", ["any", "closest", "native"])
def test_dense_equals_pairs(native, K, T, mode):
    src, snk, tris = _scene(K, T, 1000 + K + T)
    S = len(src)
    sem = native.SEM_NATIVE if mode == "native" else native.SEM_NUMBA
    bits, dist = native.visibility_dense(src, snk, tris, semantics=sem, any_hit=mode != "closest",
                                         want_dist=mode == "closest")
    s, k = np.meshgrid(np.arange(S), np.arange(K), indexing="ij")
    pairs = np.stack([s.ravel(), k.ravel() + S], 1).astype(np.int32)
    hit, d = native.raycast_pairs(np.concatenate([src, snk]), pairs, tris, semantics=sem,
                                  any_hit=mode != "closest", want_dist=mode == "closest")
    got = native.unpack_bits(bits, K)
    ref = hit.cpu().numpy().astype(bool).reshape(S, K)
    assert np.array_equal(got, ref)
    if mode == "closest":
        assert np.array_equal(dist.cpu().numpy(), d.cpu().numpy().reshape(S, K), equal_nan=True)
