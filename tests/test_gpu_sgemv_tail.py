"""fp32 products of one to eight rows whose K ends inside a chunk of 64: against float64 within the bound of any order of K fp32
additions, captured like direct, and with values that are not finite in the last rows, in their own row and column only."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# K below, at and past a lane group's 32 rows, a chunk, the sixteen chunks of one pass; N below, at and past 32 and 64 columns and
# on both sides of the wide form's 10240
SHAPES = [(1, 1, 33), (2, 7, 1), (1, 31, 64), (3, 33, 65), (8, 63, 31), (2, 65, 232), (4, 127, 100), (1, 144, 232), (8, 1023, 37),
          (5, 1025, 130), (1, 1061, 3560), (8, 133, 4045), (1, 91, 10240), (2, 200, 10243), (8, 1090, 10241)]


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_last_chunk(pkg, T, m, k, n):
    import torch
    print("sgemv tail", m, k, n, flush=True)
    rng = np.random.default_rng(m + 3 * k + 7 * n)
    a, b = (rng.normal(0, 1, s).astype(np.float32) for s in ((m, k), (k, n)))
    ta, tb = T.t(a), T.t(b)
    got = T.n(pkg.blas_matmul(ta, tb))
    want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.all(np.abs(got - want) <= k * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)))

    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        captured = pkg.blas_matmul(ta, tb)
    for _ in range(3):
        captured.zero_()
        graph.replay()
        assert np.array_equal(T.n(captured), got)

    bad_a, bad_b = a.copy(), b.copy()
    bad_a[m - 1, k - 1] = np.nan
    bad_b[k - 1, n - 1] = np.inf
    bad = T.n(pkg.blas_matmul(T.t(bad_a), T.t(bad_b)))
    assert np.all(np.isnan(bad[m - 1])) and not np.any(np.isfinite(bad[:, n - 1]))
    assert np.array_equal(bad[:m - 1, :n - 1], got[:m - 1, :n - 1])
