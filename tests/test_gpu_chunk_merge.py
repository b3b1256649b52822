"""GPU tests of the chunk merges of the field and its adjoint: source counts on both
sides of the long merge, masked, against float64 autograd."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,K", [(1, 1), (1, 17), (132, 15), (132, 16), (132, 257), (300, 2701),
                                 (2500, 31), (1100, 33),
                                 (3000, 65), (2561, 130)])
@pytest.mark.parametrize("alpha", [0.0, 0.01])
def test_chunks_against_float64(native, oracle, S, K, alpha):
    from lyceanem.differentiable import far_field

    rng = np.random.default_rng(S + K)
    pos = rng.uniform(-0.3, 0.3, (S, 3)).astype(np.float32)
    snk = rng.normal(size=(K, 3))
    snk_n = (snk / np.linalg.norm(snk, axis=1, keepdims=True)).astype(np.float32)
    snk = (30.0 * snk_n).astype(np.float32)
    w = (rng.normal(size=(S, 3)) + 1j * rng.normal(size=(S, 3))).astype(np.complex64)
    gE = (rng.normal(size=(K, 3)) + 1j * rng.normal(size=(K, 3))).astype(np.complex64)
    visible = rng.random((S, K)) < 0.7
    words = np.zeros((S, (K + 63) // 64 * 64), np.uint8)
    words[:, :K] = ~visible
    bits = torch.from_numpy(np.packbits(words, axis=1, bitorder="little").view(np.int64))
    dev, beta = native.device(), 40.0
    wd = torch.from_numpy(w).to(dev).requires_grad_(True)
    pd = torch.from_numpy(pos).to(dev).requires_grad_(True)
    E = far_field(wd, pd, torch.from_numpy(snk).to(dev), torch.from_numpy(snk_n).to(dev),
                  hit_bits=bits.to(dev), alpha=alpha, beta=beta)
    E.backward(torch.from_numpy(gE).to(dev))
    w64 = torch.from_numpy(w.astype(np.complex128)).requires_grad_(True)
    p64 = torch.from_numpy(pos.astype(np.float64)).requires_grad_(True)
    E64 = oracle.field_los_torch64(w64, p64, torch.from_numpy(snk.astype(np.float64)),
                                   torch.from_numpy(snk_n.astype(np.float64)),
                                   torch.from_numpy(visible), alpha, beta)
    E64.backward(torch.from_numpy(gE.astype(np.complex128)))
    # float32 terms of a dozen roundings each, a few of which cancel: 1e-5 of the norm is
    # some 170 of them
    for got, ref in ((E, E64), (wd.grad, w64.grad), (pd.grad, p64.grad)):
        got, ref = got.detach().cpu().numpy(), ref.detach().numpy()
        assert np.linalg.norm(got - ref) <= 1e-5 * np.linalg.norm(ref)
