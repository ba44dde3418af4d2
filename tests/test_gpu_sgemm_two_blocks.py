"""fp32 products of few rows on both sides of the lines between their kernels, and in tiles of two blocks of sixteen rows: rows, steps
and splits that do not come out even, against float64 within the bound of any order of K fp32 additions, and the same bits with B
transposed, in a group, under capture and where values of other rows are not finite."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# m, k, n: two blocks alone (the first nine) and over several workgroups (the next four); one to eight rows around 1024 k, 4096 and
# 10240 columns and whole lines of B
SHAPES = [(18, 1006, 3222), (17, 299, 3328), (26, 1328, 3072), (29, 768, 3072), (32, 768, 2304), (33, 320, 1873), (41, 968, 1952),
          (94, 321, 960), (56, 768, 1344), (94, 3048, 400), (21, 3712, 768), (90, 3055, 399), (23, 3727, 769),
          (1, 1024, 512), (1, 1088, 512), (1, 1001, 513), (8, 256, 4096), (5, 768, 4128), (5, 832, 4128), (2, 300, 4100), (3, 1061, 5120),
          (4, 1600, 10245), (4, 1601, 10245), (8, 333, 10240), (6, 255, 300),
          (8, 16, 33), (3, 15, 40), (2, 17, 4096), (5, 100, 4097), (1, 512, 90), (1, 513, 90), (1, 576, 90), (8, 512, 4128), (8, 576, 4128),
          (4, 256, 4128), (3, 320, 4128), (2, 128, 8224), (2, 192, 8224), (7, 127, 1)]


def _operands(m, k, n):
    rng = np.random.default_rng(m * 7 + k * 3 + n)
    return tuple(rng.normal(0, 1, s).astype(np.float32) for s in ((m, k), (k, n), (n,)))


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_rows_and_lines(pkg, T, m, k, n):
    import torch
    print("two blocks", m, k, n, flush=True)
    a, b, bias = _operands(m, k, n)
    flat = T.t(np.concatenate([a.ravel()[:1], a.ravel()]))[1:].view(m, k)  # rows off every 16-byte boundary
    ta, tb, tbias = T.t(a), T.t(b), T.t(bias)
    got = T.n(pkg.blas_matmul(flat, tb, tbias))
    want = a.astype(np.float64) @ b.astype(np.float64) + bias
    size = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64) + np.abs(bias)
    assert np.all(np.abs(got - want) <= (k + 1) * 2.0 ** -24 * size)
    for _ in range(3):
        assert np.array_equal(T.n(pkg.blas_matmul(ta, tb, tbias)), got)

    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        captured = pkg.blas_matmul(ta, tb, tbias)
    for _ in range(3):
        captured.zero_()
        graph.replay()
        assert np.array_equal(T.n(captured), got)

    bad = a.copy()
    bad[m // 2, k - 1] = np.inf
    rest = np.arange(m) != m // 2
    out = T.n(pkg.blas_matmul(T.t(bad), tb, tbias))
    assert np.array_equal(out[rest], got[rest]) and not np.any(np.isfinite(out[m // 2]))


@pytest.mark.parametrize("m,k,n", [(18, 1006, 3222), (41, 968, 1952), (90, 3055, 399), (8, 600, 6880), (1, 1088, 512)])
def test_transposed_and_grouped(pkg, T, m, k, n):
    a, b, bias = _operands(m, k, n)
    r = np.random.default_rng(1).normal(0, 1, (m, n)).astype(np.float32)
    outs = []
    for trans in (0, 1):
        for act in (0, 1):
            d = pkg.SgemmDesc()
            tensors = [T.t(a), T.t(np.ascontiguousarray(b.T) if trans else b), T.t(bias), T.t(r), T.t(np.zeros((m, n), np.float32))]
            d.a, d.b, d.bias, d.residual, d.c = (t.data_ptr() for t in tensors)
            d.m, d.n, d.k, d.lda, d.ldb, d.ldc = m, n, k, k, (k if trans else n), n
            d.batch_outer = d.batch_inner = 1
            d.activation, d.trans_b = act, trans
            pkg.check(pkg.lib().tfcc_rocm_sgemm_general(None, C.byref(d)))
            outs.append(T.n(tensors[4]))
    assert np.array_equal(outs[0], outs[2]) and np.array_equal(outs[1], outs[3])
    assert np.array_equal(outs[0], T.n(pkg.blas_matmul(T.t(a), T.t(b), T.t(bias))) + r)
    bs = [b, np.ascontiguousarray(b[::-1]), -b]
    for c, one in zip(pkg.sgemm_grouped(T.t(a), [T.t(x) for x in bs], [T.t(bias)] * 3), bs):
        assert np.array_equal(T.n(c), T.n(pkg.blas_matmul(T.t(a), T.t(one), T.t(bias))))
