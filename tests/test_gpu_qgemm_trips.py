"""Small quantized products whose K is shared by few workgroups of four to eight trips each: edges of tiles, K that ends inside a step,
odd addresses, both sides of the line, several calls in a row and under capture; whole numbers, so exactly the sums of 64-bit integers."""
import numpy as np
import pytest

from test_gpu_qgemm_split_k import shared_by

pytestmark = pytest.mark.gpu

# m, k, n, shared
SHAPES = [(43, 7005, 1920, True), (830, 5881, 96, True), (8, 8061, 6943, True), (1, 6692, 6603, True), (475, 6272, 152, True),
          (505, 6984, 256, True), (22, 5950, 2844, True), (1794, 5965, 96, True), (221, 4120, 1101, False), (387, 3240, 592, False)]


@pytest.mark.parametrize("m,k,n,shared", SHAPES)
def test_long_trips(pkg, T, m, k, n, shared):
    import torch
    print("trips", m, k, n, flush=True)
    assert (shared_by(m, k, n) > 1) == shared
    rng = np.random.default_rng(m + 3 * k + n)
    a, b = rng.integers(0, 256, (m, k), np.uint8), rng.integers(-128, 128, (k, n), np.int8)
    want = ((a.astype(np.float64) - 100) @ (b.astype(np.float64) + 11)).astype(np.int64)  # whole numbers below 2^53
    low_a, high_a, low_b, high_b = (T.f1(v) for v in (-100.0, 155.0, -117.0, 138.0))
    flat = T.t(np.concatenate([[0], b.reshape(-1)]).astype(np.int8))
    ta, tb = T.t(a), flat[1:].view(k, n)
    row, col = pkg.reduce_sum(ta, True), pkg.reduce_sum(T.t(b), False)
    for _ in range(3):
        acc, low, high = pkg.quantization_matmul(ta, row, low_a, high_a, tb, col, low_b, high_b)
        assert np.array_equal(T.n(acc), want)
    lo, hi = T.f1(-3e6), T.f1(3e6)
    q = pkg.quantization_matmul_requantize(ta, row, low_a, high_a, tb, col, low_b, high_b, lo, hi)[0]
    assert np.array_equal(T.n(q), T.n(pkg.requantize(acc, low, high, lo, hi, torch.uint8)))
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        captured = pkg.quantization_matmul(ta, row, low_a, high_a, tb, col, low_b, high_b)[0]
    for _ in range(3):
        captured.zero_()
        graph.replay()
        assert np.array_equal(T.n(captured), want)
