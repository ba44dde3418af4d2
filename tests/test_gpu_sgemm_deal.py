"""fp32 products whose K is dealt out over the wavefronts of one or several workgroups: tiles, steps and splits that do not come
out even, against float64 within the bound of any order of K fp32 additions, and the same bits with B transposed, in a group,
under capture and beside values that are not finite in other rows."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

# m, k, n: tiles of 32 and 64 columns, two to eight splits, K at and around whole steps, edges of tiles in both directions
SHAPES = [(75, 3072, 832), (96, 7608, 824), (24, 3183, 2827), (369, 1220, 170), (128, 2384, 992), (71, 3857, 1650), (64, 16391, 1024),
          (95, 5256, 720), (969, 7809, 72), (204, 2905, 334), (700, 2049, 90), (134, 3258, 1499), (17, 1511, 3066), (466, 5927, 289)]


def _operands(m, k, n):
    rng = np.random.default_rng(m * 7 + k * 3 + n)
    return tuple(rng.normal(0, 1, s).astype(np.float32) for s in ((m, k), (k, n), (n,)))


def _goes_there(m, k, n):
    """splits and blocks of the dispatcher's own plan (tests/cpp/sgemm_deal_plan_tests.cpp)"""
    host = os.path.join(ROOT, "wechat-tfcc_amd", "host")
    exe = os.path.join(host, "build", "sgemm_deal_plan_tests")
    if not os.path.exists(exe):
        subprocess.check_call(["make", "-C", host, "build/sgemm_deal_plan_tests"])
    return int(subprocess.check_output([exe, str(m), str(n), str(k)]).split()[0]) > 0


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_dealt_products(pkg, T, m, k, n):
    import torch
    print("dealt", m, k, n, flush=True)
    assert _goes_there(m, k, n)
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

    # what is not finite stays in its row and column
    bad = a.copy()
    bad[m // 2, k - 1] = np.inf
    rows = np.arange(m) != m // 2
    assert np.array_equal(T.n(pkg.blas_matmul(T.t(bad), tb, tbias))[rows], got[rows])


@pytest.mark.parametrize("m,k,n", [(75, 3073, 832), (96, 7608, 824), (204, 2905, 334)])
def test_dealt_products_transposed_with_residual_and_gelu(pkg, T, m, k, n):
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


def test_dealt_products_in_groups_and_on_many_streams(pkg, T):
    import torch
    a, _, _ = _operands(75, 3072, 832)
    ta = T.t(a)
    rng = np.random.default_rng(2)
    bs, biases = ([T.t(rng.normal(0, 1, s).astype(np.float32)) for _ in range(4)] for s in ((3072, 832), (832,)))
    want = [pkg.blas_matmul(ta, b, bias) for b, bias in zip(bs, biases)]
    for groups in (2, 3, 4):
        for c, w in zip(pkg.sgemm_grouped(ta, bs[:groups], biases[:groups]), want):
            assert torch.equal(c, w)
    streams = [torch.cuda.Stream() for _ in range(8)]
    torch.cuda.synchronize()
    outs = []
    for _ in range(4):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                outs.append((i % 4, pkg.blas_matmul(ta, bs[i % 4], biases[i % 4])))
    torch.cuda.synchronize()
    for i, o in outs:
        assert torch.equal(o, want[i])
