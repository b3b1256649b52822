"""CPU tests of the weight rows of MaximumDirectivityMap computed in blocks and threads:
the same bits however the rows are cut, and the caller's numpy error state."""
import numpy as np
import pytest
import torch

from lyceanem.electromagnetics import beamforming as BF


def _weights(ne, n_el, n_az, phase_resolution=24, distance=1.0):
    rng = np.random.default_rng(5)
    Et = (rng.normal(size=(ne, n_el, n_az)) + 1j * rng.normal(size=(ne, n_el, n_az)))
    Et = Et.astype(np.complex64)
    Ep = (1j * Et[::-1]).copy()
    pts = rng.normal(size=(ne, 3)) * distance
    az, el = np.linspace(-180, 180, n_az), np.linspace(-90, 90, n_el)
    return BF.command_weights(Et, Ep, pts, 0.1, az, el, np.arange(n_az)[::2], np.arange(n_el),
                              phase_resolution)


@pytest.mark.parametrize("ne,n_el,n_az", [(1, 2, 3), (9, 13, 25), (300, 21, 23), (16385, 1, 5),
                                          (257, 37, 31)])
@pytest.mark.parametrize("bits", [24, 6])
def test_blocks_and_threads_give_the_same_bits(monkeypatch, ne, n_el, n_az, bits):
    monkeypatch.setattr(torch, "get_num_threads", lambda: 1)
    monkeypatch.setattr(BF, "_BLOCK_MAX", 1 << 40)
    W0, p0 = _weights(ne, n_el, n_az, bits)
    monkeypatch.setattr(torch, "get_num_threads", lambda: 5)
    for least, most in [(BF._BLOCK_MIN, 1 << 15), (1, 1 << 15), (1000, 1001)]:
        monkeypatch.setattr(BF, "_BLOCK_MIN", least)
        monkeypatch.setattr(BF, "_BLOCK_MAX", most)
        W, p = _weights(ne, n_el, n_az, bits)
        assert W.shape == (len(range(0, n_az, 2)), n_el, 3, ne) and np.array_equal(W, W0)
        assert np.array_equal(p, p0)


def test_threads_keep_the_error_state(monkeypatch):
    monkeypatch.setattr(torch, "get_num_threads", lambda: 4)
    monkeypatch.setattr(BF, "_BLOCK_MIN", 1)
    with np.errstate(over="raise"):
        with pytest.raises(FloatingPointError):
            _weights(64, 9, 9, distance=1e200)


def test_no_commands():
    W, p = BF.command_weights(np.ones((4, 3, 5), np.complex64), np.ones((4, 3, 5), np.complex64),
                              np.zeros((4, 3)), 0.1, np.linspace(-180, 180, 5),
                              np.linspace(-90, 90, 3), np.zeros(0, int), np.zeros(0, int))
    assert W.shape == (0, 0, 3, 4) and p.shape == (0, 0, 3)
