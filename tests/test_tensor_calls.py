"""The compiled form of the operators (host/tensor_calls.cpp) takes the plain case, gives what the Python form gives bit for
bit, and declines everything else, which the Python form then sees to."""
import pytest


class Declines:
    def __getattr__(self, name):
        return lambda *args: None


def operands(torch, m, k, n):
    g = torch.Generator(device="cuda")
    g.manual_seed(m * 1000 + n)
    f = lambda *s: torch.randn(s, generator=g, device="cuda")
    a = torch.randint(0, 256, (m, k), generator=g, device="cuda", dtype=torch.uint8)
    b = torch.randint(-127, 128, (k, n), generator=g, device="cuda", dtype=torch.int8)
    return f, a, b


def test_cpu_tensors_are_declined(pkg):
    torch = pytest.importorskip("torch")
    x = torch.zeros(2, 2)
    assert pkg._native().blas_matmul(x, x, None) is None
    assert pkg._native().quantize(x, torch.uint8) is None
    assert pkg._native().reduce_sum(x.to(torch.uint8), True) is None
    assert pkg._native().blas_matmul(x, x) is None and pkg._native().dequantize(1, 2, 3) is None


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,n", [(1, 64, 48), (8, 256, 100), (3, 65, 33), (130, 96, 70)])
def test_same_bits_as_the_python_form(pkg, dev, monkeypatch, m, k, n):
    import torch
    f, a, b = operands(torch, m, k, n)
    one = lambda v: torch.tensor([v], device="cuda")
    lo, hi = one(-128.0), one(127.0)
    x, w, bias, w3 = f(m, k), f(k, n), f(n), f(5, k, n)

    def everything():
        row, col = pkg.reduce_sum(a, True), pkg.reduce_sum(b, False)
        outs = [pkg.blas_matmul(x, w), pkg.blas_matmul(x, w, bias), pkg.blas_matmul(x.expand(5, m, k).contiguous(), w3),
                pkg.blas_matmul(x.expand(4, m, k).contiguous(), w, bias), row, col]
        c, c_lo, c_hi = pkg.quantization_matmul(a, row, lo, hi, b, col, lo, hi)
        outs += [c, c_lo, c_hi, pkg.dequantize(c, c_lo, c_hi)]
        for acc in (False, True):
            for exact in (False, True):
                outs += pkg.quantization_matmul_requantize(a, row, lo, hi, b, col, lo, hi, one(-9e5), one(9e5), want_acc=acc,
                                                           colsum_exact=exact)
        if m <= 8 and k % 16 == 0:  # the packed form takes no other k
            scale = torch.rand(n, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
            for acc in (False, True):
                outs += pkg.gemv_dequant(a, b, row, col, -128, 3, 0.02, scale, want_acc=acc)
                outs += pkg.gemv_dequant(a, b, row, col, -128, 3, 0.02, scale, want_acc=acc, colsum_exact=True)
                outs += pkg.gemv_dequant_packed(a, pkg.gemv_pack(b), n, row, col, -128, 3, 0.02, scale, want_acc=acc)
        for t in (torch.uint8, torch.int8, torch.int16, torch.int32):
            outs += pkg.quantize(x, t)
        return outs

    assert pkg._native().blas_matmul(x, w, bias) is not None and pkg._native().quantize(x, torch.uint8) is not None
    compiled = everything()
    monkeypatch.setattr(pkg, "_calls", Declines())
    python = everything()
    assert len(compiled) == len(python)
    for p, q in zip(compiled, python):
        assert (p is None) == (q is None)
        if p is not None:
            assert p.dtype == q.dtype and p.shape == q.shape and torch.equal(p, q)


@pytest.mark.gpu
def test_what_is_not_plain_is_left_to_the_python_form(pkg, dev):
    import torch
    f, a, b = operands(torch, 16, 32, 24)
    x, w = f(16, 32), f(32, 24)
    native = pkg._native()
    for args in ((x[::2], w, None), (x, w.t().contiguous().t(), None), (x.double(), w, None), (x, w[:31], None), (x, w, w),
                 (f(4, 16, 32), f(1, 32, 24), None), (x[:0], w, None), (x, w.cpu(), None)):
        assert native.blas_matmul(*args) is None
    assert torch.equal(pkg.blas_matmul(x[::2], w), pkg.blas_matmul(x[::2].contiguous(), w))
    with pytest.raises(pkg.InvalidArgumentError):
        pkg.blas_matmul(x, w[:31])
    with pytest.raises(NotImplementedError):
        pkg.blas_matmul(x.double(), w)
    with pytest.raises(pkg.InvalidArgumentError):
        pkg.reduce_sum(a[:0], True)


@pytest.mark.gpu
def test_tensors_without_memory_raise(pkg, dev):
    import torch
    f, a, b = operands(torch, 8, 32, 24)
    x3, w, one = f(3, 8, 32), f(32, 24), torch.tensor([1.0], device="cuda")
    seen = []

    def mapped(call):
        def inner(t):
            seen.append(call(pkg._native(), t))
            return t
        return inner

    for x, call in ((x3, lambda n, t: n.blas_matmul(t, w, None)), (x3, lambda n, t: n.quantize(t, torch.uint8)),
                    (a.expand(3, 8, 32).contiguous(), lambda n, t: n.reduce_sum(t, True)),
                    (torch.ones((3, 8), dtype=torch.int32, device="cuda"), lambda n, t: n.dequantize(t, one, one))):
        torch.vmap(mapped(call))(x)  # the compiled form declines
    assert seen == [None] * 4
    for x, call in ((x3, lambda t: pkg.blas_matmul(t, w)), (x3, lambda t: pkg.quantize(t, torch.uint8)[0])):
        with pytest.raises(RuntimeError):  # and the Python form raises, as it cannot have their address
            torch.vmap(call)(x)
    assert torch.allclose(pkg.blas_matmul(x3, w), torch.matmul(x3, w), rtol=1e-5, atol=1e-4)  # and nothing is left behind
