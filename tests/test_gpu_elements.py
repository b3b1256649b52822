"""GPU tests of the per-element network's stores: sink counts around a wavefront and a
workgroup, one source a workgroup and several, masked and weighted, against the same
rows computed a few sources at a time; and against float64."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,K", [(16389, 1), (16384, 63), (16390, 64), (16385, 65), (8197, 300),
                                 (5500, 777)])
@pytest.mark.parametrize("tangent", [False, True])
def test_elements_many_sources(native, oracle, S, K, tangent):
    rng = np.random.default_rng(S + K)
    src = torch.from_numpy(rng.uniform(-0.3, 0.3, (S, 3)).astype(np.float32)).to(native.device())
    w = torch.from_numpy((rng.normal(size=(S, 3)) + 1j * rng.normal(size=(S, 3))).astype(
        np.complex64)).to(src.device)
    snk = rng.normal(size=(K, 3))
    n = (snk / np.linalg.norm(snk, axis=1, keepdims=True)).astype(np.float32)
    snk = (25.0 * n).astype(np.float32)
    sw = (rng.normal(size=(K, 3)) + 1j).astype(np.complex64)
    words = np.zeros((S, (K + 63) // 64 * 64), np.uint8)
    words[:, :K] = rng.random((S, K)) < 0.3
    bits = torch.from_numpy(np.packbits(words, axis=1, bitorder="little").view(np.int64)).to(
        src.device)

    def net(a, b):
        return native.field_los(src[a:b], w[a:b], snk, n, snk_w=sw, hit_bits=bits[a:b].contiguous(),
                                beta=40.0, elements=True, sink_tangent=tangent)

    got = net(0, S)
    assert got.shape == (S, K, 3)
    for a, b in ((0, 9), (4093, 4101), (S - 17, S)):
        assert torch.equal(torch.view_as_real(got[a:b]), torch.view_as_real(net(a, b)))
    blocked = torch.from_numpy(words[:, :K].astype(bool)).to(src.device)
    assert torch.all(got[blocked] == 0)
    if not tangent:
        ref = oracle.field_los(src[:9].cpu().numpy(), w[:9].cpu().numpy(), snk, n, 0.0, 40.0,
                               elements=True) * sw[None]
        ref[words[:9, :K].astype(bool)] = 0
        # a dozen float32 roundings a field
        assert np.linalg.norm(got[:9].cpu().numpy() - ref) <= 2e-6 * max(np.linalg.norm(ref), 1e-30)
