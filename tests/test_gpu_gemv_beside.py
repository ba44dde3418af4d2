"""int8 products of up to eight rows that run beside each other without a stream's order between them: two graphs recorded on one
stream and replayed on two, beside that stream's own calls, and threads on hipStreamPerThread, one handle for a stream each.  None of
them may add up the parts of K in words that another one uses.  Whole numbers, so exactly the sums of 64-bit integers."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# m, k, n: any alignment (its workspace in parts of sixteen and of eight wavefronts), aligned, aligned with a K that sixteen wavefronts
# have in one part, aligned with several steps a wavefront
SHAPES = [(3, 5748, 10293), (2, 3001, 3999), (4, 2048, 8192), (8, 4096, 2304), (4, 1024, 8192), (1, 16384, 17408)]


def _operands(T, m, k, n, count):
    rng = np.random.default_rng(m + 3 * k + 7 * n)
    b = rng.integers(-128, 128, (k, n), np.int8)
    cases = []
    for _ in range(count):
        a = rng.integers(0, 256, (m, k), np.uint8)
        cases.append((T.t(a), ((a.astype(np.float64) + 3) @ (b.astype(np.float64) - 5)).astype(np.int64)))
    return T.t(b), cases


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_graphs_of_one_stream_replayed_on_two(pkg, T, m, k, n):
    import torch
    print("gemv graphs", m, k, n, flush=True)
    tb, cases = _operands(T, m, k, n, 3)
    col, scale = pkg.reduce_sum(tb, False), torch.rand(n, device="cuda")
    rows = [pkg.reduce_sum(a, True) for a, _ in cases]

    def call(i):
        return pkg.gemv_dequant(cases[i][0], tb, rows[i], col, 3, -5, .01, scale, colsum_exact=True)[1]

    recorded, others = torch.cuda.Stream(), [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    with torch.cuda.stream(recorded):
        call(2)  # the stream has what its own calls need
    graphs, captured = [torch.cuda.CUDAGraph() for _ in range(2)], []
    torch.cuda.synchronize()
    for i, graph in enumerate(graphs):
        with torch.cuda.graph(graph, stream=recorded):
            captured.append(call(i))
    for _ in range(3):
        for c in captured:
            c.zero_()
        torch.cuda.synchronize()
        own = []
        for _ in range(10):
            for graph, other in zip(graphs, others):
                with torch.cuda.stream(other):
                    graph.replay()
            with torch.cuda.stream(recorded):
                own.append(call(2))
        torch.cuda.synchronize()
        for c, (_, want) in zip(captured, cases):
            assert np.array_equal(T.n(c), want)
        for c in own:
            assert np.array_equal(T.n(c), cases[2][1])
    del graphs, graph
    torch.cuda.synchronize()


@pytest.mark.parametrize("m,k,n", SHAPES[:5])
def test_threads_on_the_per_thread_stream(pkg, T, m, k, n):
    import torch
    print("gemv threads", m, k, n, flush=True)
    tb, cases = _operands(T, m, k, n, 4)
    col = pkg.reduce_sum(tb, False)
    rows = [pkg.reduce_sum(a, True) for a, _ in cases]
    outs = [[torch.zeros((m, n), dtype=torch.int32, device="cuda") for _ in range(20)] for _ in cases]
    torch.cuda.synchronize()
    per_thread, fn, failed = ctypes.c_void_p(2), pkg.lib().tfcc_rocm_gemv_u8s8s32, []

    def work(i):
        for out in outs[i]:
            if fn(per_thread, cases[i][0].data_ptr(), tb.data_ptr(), rows[i].data_ptr(), col.data_ptr(), 3, -5, m, n, k, out.data_ptr(), 1.0,
                  None, None):
                failed.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not failed
    for some, (_, want) in zip(outs, cases):
        for out in some:
            assert np.array_equal(T.n(out), want)


@pytest.mark.parametrize("m,k,n", [(4, 1024, 8192), (1, 944, 12800), (8, 768, 16016)])
def test_calls_without_allocation_whose_k_is_one_part(pkg, T, m, k, n):
    """They do not touch the one workspace of the entry point that allocates nothing: on two streams, without order."""
    import torch
    print("gemv one part", m, k, n, flush=True)
    tb, cases = _operands(T, m, k, n, 2)
    col, streams = pkg.reduce_sum(tb, False), [torch.cuda.Stream() for _ in range(2)]
    rows = [pkg.reduce_sum(a, True) for a, _ in cases]
    outs = [[torch.zeros((m, n), dtype=torch.int32, device="cuda") for _ in range(20)] for _ in cases]
    torch.cuda.synchronize()
    for pair in zip(*outs):
        for i, (out, stream) in enumerate(zip(pair, streams)):
            with torch.cuda.stream(stream):
                pkg.gemv_dequant(cases[i][0], tb, rows[i], col, 3, -5, 1.0, None, acc=out, no_alloc=True)
    torch.cuda.synchronize()
    for some, (_, want) in zip(outs, cases):
        for out in some:
            assert np.array_equal(T.n(out), want)
