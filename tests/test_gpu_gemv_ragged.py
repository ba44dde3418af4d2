"""int8 products of up to eight rows at any N, K and alignment, split over K: the last row and column of each operand, a K that ends in
any row of a lane's sixteen, both numbers of wavefronts, given and formed column sums, and under capture with and without a workspace.
Whole numbers, so the sums are exactly those of 64-bit integers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# m, k, n: on both sides of the least work that goes there (420 or 700 wavefronts of 64 k x 256 columns with exact sums,
# 1400 or 1900 without, 1345 k) up to sixteen wavefronts
SHAPES = [(1, 2052, 3704), (7, 1662, 4557), (3, 1200, 5789), (8, 2016, 5084), (2, 10125, 1235), (6, 6359, 2574), (4, 12288, 1101),
          (5, 4755, 4616), (1, 2897, 10788), (8, 3837, 9730), (2, 6240, 6483), (3, 5748, 10293), (4, 27000, 257), (6, 1345, 13569), (6, 1344, 13569),
          (2, 27009, 271), (1, 95744, 17), (8, 3136, 8961)]


def _operands(m, k, n):
    rng = np.random.default_rng(m + 3 * k + 7 * n)
    return rng.integers(0, 256, (m, k), np.uint8), rng.integers(-128, 128, (k, n), np.int8), rng.random(n, np.float32)


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_any_alignment(pkg, T, m, k, n):
    import torch
    print("ragged gemv", m, k, n, flush=True)
    a, b, scale = _operands(m, k, n)
    want = (a.astype(np.int64) + 3) @ (b.astype(np.int64) - 5)
    # operands that start at any byte, with what would be wrong to read on both sides
    def inside(x, before):
        flat = torch.full((x.size + before + 32,), 77, dtype=torch.uint8 if x.dtype == np.uint8 else torch.int8, device="cuda")
        view = flat[before:before + x.size].view(*x.shape)
        view.copy_(T.t(x))
        return view
    for before in (0, 1, 6):
        ta, tb, ts = inside(a, before), inside(b, before), T.t(scale)
        row, col = pkg.reduce_sum(T.t(a), True), pkg.reduce_sum(T.t(b), False)
        for exact in (True, False):
            out, acc = pkg.gemv_dequant(ta, tb, row, col, 3, -5, .01, ts, colsum_exact=exact)
            assert np.array_equal(T.n(acc), want)
            assert np.array_equal(T.n(out), (want * (np.float64(np.float32(.01)) * scale.astype(np.float64))).astype(np.float32))

    ta, tb, ts = T.t(a), T.t(b), T.t(scale)
    for warm in (True, False):  # a stream that has a workspace, and one that has none
        stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            if warm:
                pkg.gemv_dequant(ta, tb, row, col, 3, -5, .01, ts, colsum_exact=True)
            torch.cuda.synchronize()
            with torch.cuda.graph(graph, stream=stream):
                out, acc = pkg.gemv_dequant(ta, tb, row, col, 3, -5, .01, ts, colsum_exact=True)
        for _ in range(3):
            acc.zero_()
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(T.n(acc), want)
            pkg.gemv_dequant(ta, tb, row, col, 3, -5, .01, ts, colsum_exact=True)  # other work between replays
        del graph
        torch.cuda.synchronize()
