"""fp32 products of few rows: tiles, steps of K and splits that do not come out even, against float64 within the bound of
any order of K fp32 additions, and the same bits with B transposed, in a group, under capture and on more streams than
there is memory to meet in."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# m, k, n
SHAPES = [(1, 257, 3), (1, 3072, 768), (2, 1001, 1237), (4, 8192, 300), (5, 2048, 130), (8, 1537, 512), (9, 256, 1), (9, 257, 17), (16, 271, 16), (17, 272, 15), (9, 300, 130), (33, 511, 31), (64, 768, 768),
          (29, 1023, 1237), (9, 1024, 64), (16, 1537, 33), (48, 3072, 768), (31, 3079, 770), (9, 8192, 300), (200, 8191, 20),
          (2000, 300, 5), (15, 2560, 4096), (256, 288, 256),
          (1, 1024, 16), (3, 1040, 33), (2, 16384 + 13, 64), (1, 65536, 16), (7, 5133, 20), (20, 2047, 40), (12, 3600, 96)]  # 2 to 64 splits


def _within_bound(got, a, b, bias=None):
    want = a.astype(np.float64) @ b.astype(np.float64)
    size = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    if bias is not None:
        want, size = want + bias, size + np.abs(bias)
    assert np.all(np.abs(got - want) <= (a.shape[1] + 1) * 2.0 ** -24 * size)


def _operands(m, k, n):
    rng = np.random.default_rng(m * 7 + k * 3 + n)
    return tuple(rng.normal(0, 1, s).astype(np.float32) for s in ((m, k), (k, n), (n,)))


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_few_rows(pkg, T, m, k, n):
    import torch
    print("few rows", m, k, n, flush=True)
    a, b, bias = _operands(m, k, n)
    flat = T.t(np.concatenate([a.ravel()[:1], a.ravel()]))[1:].view(m, k)  # rows off every 16-byte boundary
    got = T.n(pkg.blas_matmul(flat, T.t(b), T.t(bias)))
    _within_bound(got, a, b, bias)
    for _ in range(3):
        assert np.array_equal(T.n(pkg.blas_matmul(T.t(a), T.t(b), T.t(bias))), got)

    graph, ta, tb, tbias = torch.cuda.CUDAGraph(), T.t(a), T.t(b), T.t(bias)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        captured = pkg.blas_matmul(ta, tb, tbias)
    for _ in range(3):
        captured.zero_()
        graph.replay()
        assert np.array_equal(T.n(captured), got)


@pytest.mark.parametrize("m,k,n", [(3, 1001, 65), (8, 4096, 300), (29, 768, 130), (9, 2050, 64), (40, 3072, 257)])
def test_few_rows_transposed_with_residual_and_gelu(pkg, T, m, k, n):
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
    plain = T.n(pkg.blas_matmul(T.t(a), T.t(b), T.t(bias)))
    assert np.array_equal(outs[0], plain + r)


def test_few_rows_on_many_streams(pkg, T):
    import torch
    a, b, _ = _operands(24, 4096, 512)
    ta, tb = T.t(a), T.t(b)
    want = T.n(pkg.blas_matmul(ta, tb))
    streams = [torch.cuda.Stream() for _ in range(12)]
    torch.cuda.synchronize()
    outs = []
    for _ in range(4):
        for s in streams:
            with torch.cuda.stream(s):
                outs.append(pkg.blas_matmul(ta, tb))
    torch.cuda.synchronize()
    for o in outs:
        assert np.array_equal(T.n(o), want)


def test_few_rows_in_a_group_under_capture(pkg, T):
    import torch
    a, _, _ = _operands(12, 4100, 64)
    ta = T.t(a)
    rng = np.random.default_rng(2)
    bs, biases = ([T.t(rng.normal(0, 1, s).astype(np.float32)) for _ in range(3)] for s in ((4100, 64), (64,)))
    eager, graph = pkg.sgemm_grouped(ta, bs, biases), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        captured = pkg.sgemm_grouped(ta, bs, biases)
    for _ in range(3):
        for c in captured:
            c.zero_()
        graph.replay()
        for c, e, b, bias in zip(captured, eager, bs, biases):
            assert torch.equal(c, e)
            assert torch.equal(e, pkg.blas_matmul(ta, b, bias))


def test_memory_of_a_stream_is_given_back(pkg, T):
    """more streams, one after the other, than the library gives memory to at once"""
    import torch
    lib = pkg.lib()
    a, b, _ = _operands(24, 4096, 512)
    ta, tb = T.t(a), T.t(b)
    want, out = pkg.blas_matmul(ta, tb), T.t(np.zeros((24, 512), np.float32))
    for _ in range(80):
        stream = C.c_void_p()
        pkg.check(lib.tfcc_rocm_stream_create(C.byref(stream)))
        out.zero_()
        torch.cuda.synchronize()
        pkg.check(lib.tfcc_rocm_sgemm_strided_batched(stream, ta.data_ptr(), 0, tb.data_ptr(), 0, None, out.data_ptr(), 0, 24, 512,
                                                      4096, 1))
        pkg.check(lib.tfcc_rocm_stream_synchronize(stream))
        assert np.array_equal(T.n(out), T.n(want))
        pkg.check(lib.tfcc_rocm_stream_destroy(stream))
