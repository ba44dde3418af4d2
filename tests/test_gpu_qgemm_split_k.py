"""Small quantized products whose K is shared by several workgroups per tile: the edges of the rule and of the tiles, K that
ends inside a step, operands at odd addresses, batches; several calls in a row (the memory the workgroups meet in has to be
zero again), on streams of their own and under capture, bit for bit against the oracle."""
import os
import subprocess

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def shared_by(m, k, n, batch=1):
    """The workgroups that share a tile by the launcher's own rule (tests/cpp/qgemm_small_plan_tests.cpp)."""
    host = os.path.join(ROOT, "wechat-tfcc_amd", "host")
    exe = os.path.join(host, "build", "qgemm_small_plan_tests")
    if not os.path.exists(exe):
        subprocess.check_call(["make", "-C", host, "build/qgemm_small_plan_tests"])
    return int(subprocess.check_output([exe] + [str(v) for v in (m, n, k, batch)]))


# m, k, n, batch
SHAPES = [(1, 1345, 1, 1), (3, 11304, 910, 1), (16, 1473, 65, 1), (17, 2049, 63, 1), (8, 12288, 512, 1), (92, 4184, 115, 1),
          (5, 4098, 130, 1), (32, 8191, 260, 1), (128, 8192, 512, 1), (7, 3000, 96, 5), (1, 3643, 2512, 1), (255, 1700, 70, 1)]


def _case(m, k, n, batch):
    rng = np.random.default_rng(m + 3 * k + n)
    lead = () if batch == 1 else (batch,)
    a = rng.integers(0, 256, lead + (m, k), dtype=np.uint8)
    b = rng.integers(-128, 128, lead + (k, n), dtype=np.int8)
    return a, b, O.reduce_sum(a, True), O.reduce_sum(b, False)


@pytest.mark.parametrize("m,k,n,batch", SHAPES)
def test_products_whose_k_is_shared(pkg, T, m, k, n, batch):
    assert shared_by(m, k, n, batch) > 1
    a, b, rs, cs = _case(m, k, n, batch)
    ranges = (-100.0, 155.0, -117.0, 138.0)
    want = O.qgemm(a, b, *O.qmatmul_offsets(*ranges), rs, cs)
    mn_c, mx_c = O.qmatmul_range(*ranges)
    real = O.dequantize(want, mn_c, mx_c).astype(np.float64)
    lo, hi = float(np.float32(real.min() + 0.1 * (np.ptp(real) + 1))), float(np.float32(real.max() + 1))
    want_q = O.requantize_s32_u8(want, mn_c, mx_c, lo, hi)
    r, flat = [T.f1(v) for v in ranges], T.t(np.concatenate([[0], b.reshape(-1)]).astype(np.int8))
    ta, tb = T.t(a), flat[1:].view(b.shape)
    for exact in (False, True, False):
        q, acc, got_lo, got_hi = pkg.quantization_matmul_requantize(ta, T.t(rs), r[0], r[1], tb, T.t(cs), r[2], r[3], T.f1(lo),
                                                                    T.f1(hi), want_acc=True, colsum_exact=exact)
        assert np.array_equal(T.n(acc), want) and np.array_equal(T.n(q), want_q)
        assert (float(T.n(got_lo)[0]), float(T.n(got_hi)[0])) == (mn_c, mx_c)
        c, _, _ = pkg.quantization_matmul(ta, T.t(rs), r[0], r[1], T.t(b), T.t(cs), r[2], r[3])
        assert np.array_equal(T.n(c), want)


@pytest.mark.parametrize("m,k,n", [(8, 12288, 512), (1, 6160, 100), (3, 11304, 910), (6, 3104, 3586)])
def test_dequantized_on_streams_and_under_capture(pkg, T, m, k, n):
    import torch
    a, b, rs, cs = _case(m, k, n, 1)
    scale = np.random.default_rng(k).uniform(0.001, 0.01, n).astype(np.float32)
    want = O.qgemm(a, b, -57, 93, rs, cs)
    want_f = (want.astype(np.float64) * (np.float64(np.float32(0.02)) * scale.astype(np.float64))).astype(np.float32)
    args = (T.t(a), T.t(b), T.t(rs), T.t(cs), -57, 93, 0.02, T.t(scale))
    streams, outs = [torch.cuda.Stream() for _ in range(6)], []
    torch.cuda.synchronize()
    for i in range(3):
        for s in streams:
            with torch.cuda.stream(s):
                outs.append(pkg.gemv_dequant(*args, colsum_exact=i == 1))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = pkg.gemv_dequant(*args)
    for _ in range(3):
        for c in captured:
            c.zero_()
        graph.replay()
        outs.append(tuple(c.clone() for c in captured))
        outs.append(pkg.gemv_dequant(*args))
    torch.cuda.synchronize()
    for f, acc in outs:
        assert np.array_equal(T.n(acc), want) and np.array_equal(T.n(f).view(np.uint32), want_f.view(np.uint32))


@pytest.mark.parametrize("m,k,n,shared", [(133, 2187, 1144, 3), (105, 2452, 25, 7), (36, 2486, 467, 7), (526, 1832, 400, 1),
                                          (1869, 1824, 32, 1), (250, 1624, 200, 1), (48, 1920, 4992, 1)])
def test_both_sides_of_the_line(pkg, T, m, k, n, shared):
    assert shared_by(m, k, n) == shared
    a, b, rs, cs = _case(m, k, n, 1)
    ranges = (-100.0, 155.0, -117.0, 138.0)
    r = [T.f1(v) for v in ranges]
    got, _, _ = pkg.quantization_matmul(T.t(a), T.t(rs), r[0], r[1], T.t(b), T.t(cs), r[2], r[3])
    assert np.array_equal(T.n(got), O.qgemm(a, b, *O.qmatmul_offsets(*ranges), rs, cs))
