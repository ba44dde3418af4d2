"""fp32 products on the bf16 matrix cores (operands split into three exact parts) at the sizes where they can go wrong: the
edges of their tiles in every direction, K that ends inside a slab, operands at odd addresses, fused epilogues, B handed over
transposed, and the values that the split cannot represent, which a tile has to notice."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 256 x 256, 128 x 128 and 64 x 64 tiles (the last with four K groups): whole tiles, one row, column or k more and less
SHAPES = [(4096, 4096, 130), (4097, 3841, 144), (3900, 4095, 255), (2048, 2048, 256), (2047, 1921, 1009), (1350, 5253, 336),
          (385, 2050, 2048), (768, 1024, 1025), (449, 1217, 2053), (2049, 769, 800), (64, 8200, 2048), (3000, 4100, 128),
          (441, 2303, 2053), (1024, 1024, 2048), (1020, 1022, 2050), (1616, 1219, 1167)]


def bound(k):
    """Of the relative 2-norm error: each of the k / 16 x 6 additions to an accumulator rounds by at most 2^-24 of the partial
    sum, independent of one another; twice their root sum of squares."""
    return 2 * (6 * k / 16) ** 0.5 * 2.0 ** -24


def rel(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_against_float64_and_the_transposed_form(pkg, dev, m, n, k):
    import torch
    gen = torch.Generator(device=dev).manual_seed(m + n + k)
    a = torch.randn(m * k + 1, device=dev, generator=gen)[1:].view(m, k)  # an odd address
    b = torch.randn(k, n, device=dev, generator=gen)
    want = a.double() @ b.double()
    out = pkg.blas_matmul(a, b)
    assert rel(out, want) <= bound(k)
    c = torch.full((m, n + 3), float("nan"), device=dev)
    pkg.sgemm_general(a, b.t().contiguous(), c, m, n, k, k, k, n + 3, trans_b=True)
    assert torch.equal(c[:, :n], out) and bool(torch.isnan(c[:, n:]).all())


@pytest.mark.parametrize("m,n,k", [(2048, 2052, 200), (1100, 2700, 300), (600, 1500, 1100), (4096, 4000, 160), (4000, 4095, 512),
                                   (2048, 2047, 1024), (1020, 1022, 2050)])
def test_bias_residual_and_gelu(pkg, dev, m, n, k):
    import torch
    gen = torch.Generator(device=dev).manual_seed(m)
    a, b, r = (torch.randn(*s, device=dev, generator=gen) for s in ((m, k), (k, n), (m, n)))
    bias = torch.randn(n, device=dev, generator=gen)
    out = torch.empty(m, n, device=dev)
    pkg.check(pkg.lib().tfcc_rocm_sgemm_fused(None, a.data_ptr(), m * k, b.data_ptr(), k * n, bias.data_ptr(), r.data_ptr(), m * n,
                                              out.data_ptr(), m * n, m, n, k, 1, 1))
    x = a.double() @ b.double() + bias.double() + r.double()
    assert rel(out, 0.5 * x * (1 + torch.erf(x / 2 ** 0.5))) <= bound(k) + 1e-6  # GELU itself: 1e-6


@pytest.mark.parametrize("m,n,k", [(2048, 2048, 256), (1350, 5253, 300), (800, 1280, 1040), (1020, 1022, 2050)])
def test_values_the_split_cannot_represent(pkg, dev, m, n, k):
    import torch
    gen = torch.Generator(device=dev).manual_seed(n)
    a = torch.randn(m, k, device=dev, generator=gen)
    b = torch.randn(k, n, device=dev, generator=gen)
    a[70] = 0.0                                  # a row of zeros, nothing wrong with it
    a[1, 5], a[2, 7] = float("inf"), float("nan")
    a[3] = 0.0
    a[3, 9], a[3, 11] = 3.3999e38, -3.3999e38    # rounds up to infinity in bf16
    b[9, :], b[11, :] = 0.25, 0.125
    a[200:204] = 0.0
    a[200, 3], b[3, :] = 2.0 ** -140, 2.0 ** 100       # subnormal next to a large partner
    a[201, 4], b[4, :] = 1.9999999 * 2.0 ** -115, 2.0  # no room for the third part
    a[202, 6], b[6, :] = 1.2345678 * 2.0 ** -70, 1.7654321 * 2.0 ** -70  # a subnormal result
    a[203, 8], b[8, :] = 1.5, 1.0
    rest = [i for i in range(m) if i not in (1, 2, 200)]
    a[rest, 3] = 0.0
    out = pkg.blas_matmul(a, b)
    want = a.double() @ b.double()
    assert torch.equal(torch.isnan(out), torch.isnan(want.float())) and torch.equal(torch.isinf(out), torch.isinf(want.float()))
    assert torch.equal(out[70], torch.zeros_like(out[70])) and torch.equal(out[203], torch.full_like(out[203], 1.5))
    exact = want[200:203].float()
    assert torch.equal(out[200:202], exact[:2]) and bool(((out[202].double() - want[202]).abs() <= 2.0 ** -149).all())
    assert rel(out[3], want[3]) <= 2.0 ** -23
    plain = [i for i in rest if i not in (3, 70) and not 200 <= i < 204]
    assert rel(out[plain], want[plain]) <= bound(k) * 2  # tiles with a bad value: fp32 matrix ops, one addition for two k


def test_results_that_cancel(pkg, dev):
    """A few results that are zero among large ones are summed again, with their bias and activation."""
    import torch
    m, n, k = 2048, 2048, 256
    gen = torch.Generator(device=dev).manual_seed(3)
    a = torch.randn(m, k, device=dev, generator=gen)
    b = torch.randn(k, n, device=dev, generator=gen)
    a[100, 1::2] = a[100, 0::2]
    b[1::2, 33] = -b[0::2, 33]
    b[1::2, 1999] = -b[0::2, 1999]
    bias = torch.randn(n, device=dev, generator=gen)
    out = pkg.blas_matmul(a, b, bias)
    assert rel(out, a.double() @ b.double() + bias.double()) <= bound(k)
    # sums of pairs that cancel exactly in any order of fp32 additions that keeps the pairs, and nearly in the others
    assert abs(out[100, 33] - bias[33]) < 1e-4 and abs(out[100, 1999] - bias[1999]) < 1e-4
    a[100] = 0.0
    a[100, 7], a[100, 8] = 1.0, 1.0
    b[7, 40], b[8, 40] = 3.0, -3.0
    out = pkg.blas_matmul(a, b, bias)
    assert out[100, 40] == bias[40]
    assert rel(out, a.double() @ b.double() + bias.double()) <= bound(k)


@pytest.mark.parametrize("place", [0, 5, 134, 255])
@pytest.mark.parametrize("m,n,k", [(2048, 2048, 256), (1020, 1022, 2050)])
def test_an_operand_below_the_pieces_range_at_any_place(pkg, dev, m, n, k, place):
    """One subnormal operand, wherever it lies in its four, next to a large partner: the only thing wrong with its tile."""
    import torch
    gen = torch.Generator(device=dev).manual_seed(place)
    a, b = torch.randn(m, k, device=dev, generator=gen), torch.randn(k, n, device=dev, generator=gen)
    a[:, place], b[place, :] = 0.0, 2.0 ** 100
    a[200] = 0.0
    a[200, place] = 2.0 ** -140
    assert torch.equal(pkg.blas_matmul(a, b)[200], torch.full((n,), 2.0 ** -40, device=dev))
    a, b = b.t().contiguous(), a.t().contiguous()  # and in B, as stored and transposed
    assert torch.equal(pkg.blas_matmul(a, b)[:, 200], torch.full((n,), 2.0 ** -40, device=dev))
    c = torch.empty(n, m, device=dev)
    pkg.sgemm_general(a, b.t().contiguous(), c, n, m, k, k, k, m, trans_b=True)
    assert torch.equal(c[:, 200], torch.full((n,), 2.0 ** -40, device=dev))
