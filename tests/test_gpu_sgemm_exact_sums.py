"""fp32 products whose sums are exact in any order: odd whole numbers of at most seven, so that every partial sum is a whole number below
2^24, against int64 for equality.  No operand is zero, so a k that is left out, taken twice or paired with another one shows, however long
K is.  Products with a dealt K, of one and of two row blocks, and streamed ones, launched and replayed; and that the last k of a row, and
of a column, reaches all of its results."""
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT, rel_fro

pytestmark = pytest.mark.gpu

# m, k, n
DEALT = [(75, 3072, 832), (96, 7608, 824), (24, 3183, 2827), (369, 1220, 170), (128, 2384, 992), (71, 3857, 1650), (128, 16391, 800),
         (95, 5256, 720), (896, 5405, 120), (204, 2905, 334), (700, 2049, 90), (64, 16391, 1120), (17, 1511, 3066), (466, 5927, 289)]
FEW_ROWS = [(18, 1006, 3222), (17, 299, 3328), (41, 968, 1952), (94, 3048, 400), (90, 3055, 399), (23, 3727, 769), (9, 8192, 300), (1, 1088, 512),
            (3, 1061, 5120), (8, 16, 33), (2, 16397, 64), (1, 65536, 16), (7, 5133, 20), (211, 1903, 192),
            (64, 16391, 1024), (969, 7809, 72), (8, 1090, 10241), (2, 65, 10243), (3, 33, 10240)]
STREAMED = [(1, 960, 128), (1, 1472, 64), (2, 1216, 640), (8, 1601, 10241), (2, 1061, 5120), (4, 1601, 10272), (1, 15, 100),
            (1, 5120, 5120), (2, 2048, 3840)]


def _goes_to(m, k, n):
    """the kernel of the dispatcher's own rule (tests/cpp/sgemm_skinny_plan_tests.cpp)"""
    host = os.path.join(ROOT, "wechat-tfcc_amd", "host")
    exe = os.path.join(host, "build", "sgemm_skinny_plan_tests")
    if not os.path.exists(exe):
        subprocess.check_call(["make", "-C", host, "build/sgemm_skinny_plan_tests"])
    return subprocess.check_output([exe, str(m), str(k), str(n)], text=True).split()[0]


@pytest.mark.parametrize("kernel,m,k,n", [("deal", *s) for s in DEALT] + [("skinny", *s) for s in FEW_ROWS] + [("other", *s) for s in STREAMED])
def test_exact_sums(pkg, T, kernel, m, k, n):
    import torch
    print("exact sums", kernel, m, k, n, flush=True)
    assert _goes_to(m, k, n) == kernel
    rng = np.random.default_rng(m + 5 * k + 11 * n)
    a, b, bias = (2 * rng.integers(-4, 4, s) + 1 for s in ((m, k), (k, n), (n,)))
    want = (a.astype(np.float64) @ b.astype(np.float64) + bias).astype(np.int64)  # whole numbers below 2^24
    ta, tb, tbias = (T.t(x.astype(np.float32)) for x in (a, b, bias))
    assert np.array_equal(T.n(pkg.blas_matmul(ta, tb, tbias)), want)

    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        captured = pkg.blas_matmul(ta, tb, tbias)
    for _ in range(3):
        captured.zero_()
        graph.replay()
        assert np.array_equal(T.n(captured), want)

    # the last k of one row and of one column: theirs is not finite, the rest is as it was
    row, col = m // 2, n - 1
    ta[row, k - 1] = float("inf")
    tb[k - 1, col] = float("nan")
    out = T.n(pkg.blas_matmul(ta, tb, tbias))
    assert not np.any(np.isfinite(out[row])) and np.all(np.isnan(out[:, col]))
    rest = np.ix_(np.arange(m) != row, np.arange(n) != col)
    assert np.array_equal(out[rest], want[rest])


@pytest.mark.parametrize("m,k,n", [(75, 4928, 1344), (128, 3072, 768), (96, 7608, 824)])
def test_error_of_a_dealt_k(pkg, T, m, k, n):
    """1.2e-7 of the size of the result is what the short chains are said to leave, where four K groups leave four times that; twice as much
    is allowed."""
    assert _goes_to(m, k, n) == "deal"
    rng = np.random.default_rng(k)
    a, b = (rng.normal(0, 1, s).astype(np.float32) for s in ((m, k), (k, n)))
    assert rel_fro(T.n(pkg.blas_matmul(T.t(a), T.t(b))), a.astype(np.float64) @ b.astype(np.float64)) <= 2.4e-7
