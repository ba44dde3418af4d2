"""The edges of the quantization kernels: whole tensors in one launch and the launch behind its limit, elements behind the
last 16-byte piece, rows that start at any address.  Whole numbers and one fixed expression of floats: exact."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

LIMIT = 128 * 1024  # elements that every workgroup reads for the range where a launch is recorded (40 K otherwise)
TOGETHER = 8 << 20   # elements whose range the workgroups of one launch agree on; more take a launch for it


@pytest.mark.parametrize("total", [1, 2, 3, 5, 4095, 4096, 4097, 32771, LIMIT - 1, LIMIT, LIMIT + 1, LIMIT + 4])
@pytest.mark.parametrize("dtype", ["uint8", "int8"])
@pytest.mark.parametrize("skip", [0, 1])
def test_quantize_with_the_range_of_the_data(pkg, T, total, dtype, skip):
    import torch
    x = np.random.default_rng(total).normal(0.1, 2.0, total + skip).astype(np.float32)
    x[skip + total // 2] = 17.0  # the extremes: inside, and the very last element
    x[-1] = -31.0
    q, mn, mx = pkg.quantize(T.t(x)[skip:], getattr(torch, dtype))  # skip: not on a 16-byte boundary
    lo, hi = float(x[skip:].min()), float(x[skip:].max())
    assert (float(T.n(mn)[0]), float(T.n(mx)[0])) == (lo, hi)
    assert np.array_equal(T.n(q), O.quantize(x[skip:], lo, hi, dtype))


@pytest.mark.parametrize("total", [40960, 40961, 45057, (1 << 20) - 3, (1 << 20) + 1, (2 << 20) + 2, (4 << 20) + 3, 8 << 20, (8 << 20) + 1])
@pytest.mark.parametrize("dtype,middle", [("uint8", 0.1), ("int8", -300.0), ("int16", 1.0), ("int32", 0.0), ("uint8", 3e6)])
def test_quantize_in_workgroups_that_agree_on_the_range(pkg, T, total, dtype, middle):
    """one, two, four and eight pieces to a thread, whole numbers that fit 32 bits and that do not, a NaN and the extremes in
    the first and the last workgroup"""
    import torch
    x = np.random.default_rng(total).normal(middle, 2.0, total).astype(np.float32)
    x[3], x[-1], x[total // 3] = middle + 17.0, middle - 31.0, np.nan
    q, mn, mx = pkg.quantize(T.t(x), getattr(torch, dtype))
    lo, hi = float(np.nanmin(x)), float(np.nanmax(x))
    assert (float(T.n(mn)[0]), float(T.n(mx)[0])) == (lo, hi)
    given = O.quantize(x, lo, hi, dtype) if "int8" in dtype else T.n(pkg.quantize(T.t(x), getattr(torch, dtype), T.f1(lo), T.f1(hi)))
    assert np.array_equal(T.n(q), given)


@pytest.mark.parametrize("total", [5, 4095, 40001, LIMIT + 4])
def test_quantize_over_its_own_input(pkg, T, total):
    import torch
    x = np.random.default_rng(total).normal(0.1, 2.0, total).astype(np.float32)
    data, lo, hi = T.t(x), T.f1(0.0), T.f1(0.0)
    pkg.check(pkg.lib().tfcc_rocm_quantize_minmax(pkg._stream(), pkg._ptr(data), total, pkg._ptr(data), pkg._type_code(torch.int32),
                                                  pkg._ptr(lo), pkg._ptr(hi)))
    assert (float(T.n(lo)[0]), float(T.n(hi)[0])) == (float(x.min()), float(x.max()))
    assert np.array_equal(T.n(data).view(np.int32), T.n(pkg.quantize(T.t(x), torch.int32, lo, hi)))


@pytest.mark.parametrize("special", [[np.nan, 1.0, -2.0], [np.inf, 1.0, -2.0], [3.0, 3.0, 3.0], [np.nan] * 3, [-7.5, 0.3, 9.25]])
@pytest.mark.parametrize("dtype", ["uint8", "int16", "int32"])
def test_quantize_small_and_large_tensors_agree(pkg, T, special, dtype):
    import torch
    small = np.array(special, np.float32)
    large = np.tile(small, LIMIT // 3 + 1)  # in workgroups that agree on the range
    a, b = (pkg.quantize(T.t(v), getattr(torch, dtype)) for v in (small, large))
    for v, w in zip(a[1:], b[1:]):
        assert np.array_equal(T.n(v), T.n(w), equal_nan=True)
    assert np.array_equal(np.tile(T.n(a[0]), LIMIT // 3 + 1), T.n(b[0]))


@pytest.mark.parametrize("total", [1, 3, 4, 1023, 4097, 95249])
def test_dequantize_behind_the_last_piece(pkg, T, total):
    x = np.random.default_rng(total).integers(-2 ** 31, 2 ** 31, total, dtype=np.int64).astype(np.int32)
    got = T.n(pkg.dequantize(T.t(x), T.f1(-3.25), T.f1(7.5)))
    assert np.array_equal(got, O.dequantize(x, -3.25, 7.5))


@pytest.mark.parametrize("col", [1, 15, 16, 17, 127, 1001, 8192, 8209])
@pytest.mark.parametrize("dtype", ["uint8", "int8", "int16"])
def test_row_sums_at_any_address(pkg, T, col, dtype):
    info = np.iinfo(dtype)
    a = np.random.default_rng(col).integers(info.min, info.max + 1, (7, col)).astype(dtype)
    flat = T.t(np.concatenate([a[0, :1], a.ravel()]))
    for t in (T.t(a), flat[1:].view(7, col)):
        assert np.array_equal(T.n(pkg.reduce_sum(t, True)).ravel(), a.sum(1, dtype=np.int64).astype(np.int32))


@pytest.mark.parametrize("total", [3 * LIMIT, TOGETHER + 4])
def test_quantize_on_several_streams_and_under_capture(pkg, T, total):
    """the words of the workgroups that agree on the range, and behind those the arrival words of a stream, side by side"""
    import torch
    rng = np.random.default_rng(3)
    xs = [rng.normal(0, 1 + i, total + i).astype(np.float32) for i in range(4)]
    ts, streams = [T.t(x) for x in xs], [torch.cuda.Stream() for _ in xs]
    torch.cuda.synchronize()
    want = [O.quantize(x, float(x.min()), float(x.max()), "uint8") for x in xs]
    outs = []
    for _ in range(5):
        for t, s in zip(ts, streams):
            with torch.cuda.stream(s):
                outs.append(pkg.quantize(t, torch.uint8)[0])
    torch.cuda.synchronize()
    for i, q in enumerate(outs):
        assert np.array_equal(T.n(q), want[i % 4])
    graph, static = torch.cuda.CUDAGraph(), ts[0].clone()
    with torch.cuda.graph(graph):
        q = pkg.quantize(static, torch.uint8)[0]
    for i in (0, 0, 0):
        static.copy_(ts[i])
        graph.replay()
        eager = pkg.quantize(ts[1], torch.uint8)[0]
        torch.cuda.synchronize()
        assert np.array_equal(T.n(q), want[0]) and np.array_equal(T.n(eager), want[1])
        q.zero_()


@pytest.mark.parametrize("total", [3 << 20, TOGETHER])
def test_large_tensors_of_several_streams(pkg, T, total):
    """Launches whose workgroups all wait for one another do not fit the GPU side by side: on four streams a call takes no longer than
    on one (us, on one / on four: 3 M 8.6 / 8.5, 8 M 13.1 / 14.4; all four in one launch each 13.8 and 27; the line lies at half as much again)"""
    import time
    import torch
    xs = [torch.randn(total, device="cuda") for _ in range(4)]
    many = [torch.cuda.Stream() for _ in xs]
    want = [O.quantize(T.n(x), float(x.min()), float(x.max()), "uint8") for x in xs]

    def best(streams):
        times = []
        for _ in range(7):
            torch.cuda.synchronize()
            start = time.perf_counter()
            for _ in range(20):
                for x, s, q, ends in zip(xs, streams, qs, ranges):
                    pkg.check(pkg.lib().tfcc_rocm_quantize_minmax(s.cuda_stream, pkg._ptr(x), total, pkg._ptr(q), pkg._type_code(torch.uint8),
                                                                  pkg._ptr(ends[:1]), pkg._ptr(ends[1:])))
            torch.cuda.synchronize()
            times.append(time.perf_counter() - start)
        return min(times)

    qs, ranges = [torch.empty(total, dtype=torch.uint8, device="cuda") for _ in xs], [torch.empty(2, device="cuda") for _ in xs]
    one, four = best(many[:1] * 4), best(many)
    for q, w in zip(qs, want):
        assert np.array_equal(T.n(q), w)
    assert four <= 1.5 * one


@pytest.mark.parametrize("total", [LIMIT + 1, LIMIT + 16384, 64 * 16384 + 3, 256 * 16384 - 1, 256 * 16384 + 5, 16 << 20])
def test_captured_quantize_of_the_data_s_own_range(pkg, T, total):
    """Recorded in a graph: the same bytes as outside, and no slower than a launch more (with an atomic per wavefront on the
    two results 16 M elements took twelve times as long).  A replay of three launches takes 20 to 50 us whatever they do, most
    of it the host's, and now and then twice that; so two such replays of launches that do nothing are added to the bound."""
    import torch
    x = np.random.default_rng(total).normal(0.0, 3.0, total).astype(np.float32)
    x[0], x[-1] = -40.0, 41.0
    t, graph = T.t(x), torch.cuda.CUDAGraph()
    want = O.quantize(x, -40.0, 41.0, "uint8")
    eager = pkg.quantize(t, torch.uint8)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        captured = pkg.quantize(t, torch.uint8)
    for _ in range(3):
        for c in captured:
            c.zero_()
        graph.replay()
        for c, e in zip(captured, eager):
            assert torch.equal(c, e)
        assert np.array_equal(T.n(captured[0]), want)

    idle, one = torch.cuda.CUDAGraph(), torch.zeros(1, device="cuda")
    with torch.cuda.graph(idle):
        for _ in range(3):
            one.zero_()

    def best(f):
        times = []
        for _ in range(15):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            f()
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end) * 1e3)
        return min(times)

    assert best(graph.replay) <= 2.0 * best(lambda: pkg.quantize(t, torch.uint8)) + 2.0 * best(idle.replay)


@pytest.mark.parametrize("total", [40961, (1 << 20) - 3, (2 << 20) + 2, (4 << 20) + 3, 8 << 20])
@pytest.mark.parametrize("wait_us", [0, 1])
def test_quantize_whose_workgroups_do_not_wait(pkg, T, total, wait_us):
    """a workgroup that has waited long enough finds the range of the parts that are missing itself: one, two, four and eight
    pieces to a thread, the extremes and a NaN in the first and the last part"""
    import torch
    x = np.random.default_rng(total).normal(0.1, 2.0, total).astype(np.float32)
    x[5], x[-1], x[total // 2] = 17.0, -31.0, np.nan
    data, want = T.t(x), O.quantize(x, -31.0, 17.0, "uint8")
    for _ in range(3):
        q, low, high = torch.zeros(total, dtype=torch.uint8, device="cuda"), T.f1(0.0), T.f1(0.0)
        pkg.check(pkg.lib().tfcc_rocm_quantize_minmax_wait(pkg._stream(), pkg._ptr(data), total, pkg._ptr(q), pkg._type_code(torch.uint8),
                                                           pkg._ptr(low), pkg._ptr(high), wait_us))
        assert (float(T.n(low)[0]), float(T.n(high)[0])) == (-31.0, 17.0)
        assert np.array_equal(T.n(q), want)
