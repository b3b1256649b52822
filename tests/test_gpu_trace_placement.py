"""GPU tests of the trace's placement by buckets: chunk, bucket and sample edges,
skewed starts, against float64 sums; and the longest traces, which sort."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(amp, bins, exc, N):
    b = np.maximum(bins, 0)
    ok = b < N
    H, A = np.zeros((N, 3)), np.zeros((N, 3))
    np.add.at(H, b[ok], amp[ok])
    np.add.at(A, b[ok], np.abs(amp[ok]))
    out, mag = np.zeros((N, 3)), np.zeros((N, 3))
    for j in range(min(len(exc), N)):
        out[j:] += exc[j] * H[:N - j]
        mag[j:] += abs(exc[j]) * A[:N - j]
    return out, mag


@pytest.mark.parametrize("N", [1, 255, 256, 257, 1024, 1025, 65536, 65537, 262144, 262145])
@pytest.mark.parametrize("V", [1, 63, 2048, 2049, 20000, 140000])
def test_trace_buckets(native, N, V):
    rng = np.random.default_rng(N + V)
    amp = rng.normal(size=(V, 3)) * 10.0 ** rng.integers(-6, 3, (V, 1))
    for kind in range(4):
        if kind == 0:    # over the trace and past both ends
            bins = rng.integers(-N // 4 - 1, N + N // 4 + 2, V)
        elif kind == 1:  # one sample
            bins = np.full(V, N // 2)
        elif kind == 2:  # two neighbours and the last, sorted
            bins = np.sort(rng.choice([0, min(1, N - 1), N - 1], V))
        else:            # none
            bins = np.full(V, N)
        exc = rng.normal(size=5)
        got = native.time_trace(amp, bins, exc, N).cpu().numpy()
        again = native.time_trace(amp, bins, exc, N).cpu().numpy()
        ref, mag = _reference(amp, bins, exc, N)
        assert np.array_equal(got, again)
        # both orders of at most V + 5 additions: V 2^-52 of the sum of magnitudes is
        # far above what roundings of random sign reach
        assert np.all(np.abs(got - ref) <= (V + 10) * 2.0 ** -52 * mag)


def test_trace_values_that_are_not_finite(native):
    """They stay in their own sample; starts that are not numbers are past the end."""
    rng = np.random.default_rng(3)
    V, N = 5000, 3000
    amp, bins = rng.normal(size=(V, 3)), rng.integers(0, N, V)
    amp[7], amp[4000, 1] = np.nan, np.inf
    got = native.time_trace(amp, bins, [1.0], N).cpu().numpy()
    ref, _ = _reference(amp, bins, [1.0], N)
    assert np.array_equal(np.isfinite(got), np.isfinite(ref))
    ok = np.isfinite(ref)
    assert np.allclose(got[ok], ref[ok], rtol=0, atol=1e-12)


def test_trace_in_a_graph(native):
    """Replays of the captured placement follow the inputs."""
    rng = np.random.default_rng(4)
    V, N = 30000, 5000
    lib = native.load_library()
    dev = native.device()
    amp = torch.empty((V, 3), dtype=torch.float64, device=dev)
    bins = torch.empty(V, dtype=torch.int64, device=dev)
    exc = torch.tensor([1.0, -0.5, 0.25], dtype=torch.float64, device=dev)
    out = torch.empty((N, 3), dtype=torch.float64, device=dev)
    wsb = int(lib.lem_time_trace_workspace(V, N))
    ws = torch.empty(wsb, dtype=torch.uint8, device=dev)

    def step():
        native.check(lib.lem_time_trace(native.ptr(amp), native.ptr(bins), V, native.ptr(exc), 3,
                                        N, native.ptr(out), native.ptr(ws), wsb,
                                        native.stream_ptr()), "lem_time_trace")

    def fill():
        a, b = rng.normal(size=(V, 3)), rng.integers(-5, N + 50, V)
        amp.copy_(torch.from_numpy(a))
        bins.copy_(torch.from_numpy(b))
        return _reference(a, b, exc.cpu().numpy(), N)

    fill()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for _ in range(4):
        ref, mag = fill()
        graph.replay()
        torch.cuda.synchronize()
        assert np.all(np.abs(out.cpu().numpy() - ref) <= 100 * 2.0 ** -52 * mag)
