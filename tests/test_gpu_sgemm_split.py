"""fp32 products on the bf16 matrix cores (operands split into three exact parts) at the sizes where they can go wrong: the
edges of their tiles in every direction, K that ends inside a slab, operands at odd addresses, fused epilogues, B handed over
transposed, and the values that the split cannot represent, which a tile has to notice."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NONE, WIDE, K128, K64 = -1, 0, 1, 2  # tiles of 128 x 256, 128 x 128, 64 x 64 (with four K groups); NONE: the fp32 matrix ops


def kernel_of(m, n, k, batch=1):
    """The kernel that the dispatcher's own rule picks (tests/cpp/sgemm_split_plan_tests.cpp)."""
    host = os.path.join(ROOT, "wechat-tfcc_amd", "host")
    exe = os.path.join(host, "build", "sgemm_split_plan_tests")
    if not os.path.exists(exe):
        subprocess.check_call(["make", "-C", host, "build/sgemm_split_plan_tests"])
    return int(subprocess.check_output([exe] + [str(v) for v in (m, n, k, batch)]))


# whole tiles, one row, column or k more and less, K that ends inside a slab, the shortest K, few rows, few columns
SHAPES = [(WIDE, 4096, 4096, 512), (WIDE, 3969, 3841, 600), (WIDE, 3900, 4095, 511), (WIDE, 1350, 5253, 336), (WIDE, 833, 4976, 616),
          (WIDE, 2954, 1353, 1013), (WIDE, 2048, 4096, 1025),
          (K128, 4096, 4096, 130), (K128, 4097, 3841, 144), (K128, 2048, 2048, 256), (K128, 2047, 1921, 1009), (K128, 3000, 4100, 128),
          (K128, 544, 4924, 478), (K128, 2904, 938, 441), (K128, 2992, 2020, 129),
          (K64, 441, 2303, 2053), (K64, 1024, 1024, 2048), (K64, 1020, 1022, 2050), (K64, 2476, 3285, 395), (K64, 2199, 3656, 414),
          (K64, 415, 4495, 1093), (K64, 2912, 656, 1009), (K64, 256, 6593, 1800),
          # on the other side of the line
          (NONE, 385, 2050, 2048), (NONE, 768, 1024, 1025), (NONE, 449, 1217, 2053), (NONE, 2049, 769, 800), (NONE, 64, 8200, 2048),
          (NONE, 1616, 1219, 1167)]
ONE_OF_EACH = [(WIDE, 2048, 4096, 1025), (K128, 2047, 1921, 1009), (K64, 1020, 1022, 2050)]


def bound(k):
    """Of the relative 2-norm error.  k / 16 additions to the large accumulator, each rounded by at most 2^-24 of a partial sum
    and independent of one another, and the one that joins the two; the small terms are rounded 2^8 below that.  (A term
    that is left out shows as 2.4e-6.)"""
    return 2.0 ** -24 * (1 + (k / 16) ** 0.5)


def bound_fp32(k):
    """The same for k / 2 additions, as the fp32 matrix ops make them, or six for every 16 k, and twice that."""
    return 2 * (6 * k / 16) ** 0.5 * 2.0 ** -24


def rel(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("kernel,m,n,k", SHAPES)
def test_against_float64_and_the_transposed_form(pkg, dev, kernel, m, n, k):
    import torch
    assert kernel_of(m, n, k) == kernel
    gen = torch.Generator(device=dev).manual_seed(m + n + k)
    a = torch.randn(m * k + 1, device=dev, generator=gen)[1:].view(m, k)  # an odd address
    b = torch.randn(k, n, device=dev, generator=gen)
    want = a.double() @ b.double()
    out = pkg.blas_matmul(a, b)
    print(kernel, rel(out, want), bound(k))
    assert rel(out, want) <= (bound(k) if kernel != NONE else bound_fp32(k))
    c = torch.full((m, n + 3), float("nan"), device=dev)
    pkg.sgemm_general(a, b.t().contiguous(), c, m, n, k, k, k, n + 3, trans_b=True)
    assert torch.equal(c[:, :n], out) and bool(torch.isnan(c[:, n:]).all())


@pytest.mark.parametrize("m,n,k", [(2048, 2048, 320), (2047, 2041, 321), (1921, 2048, 335), (2048, 1930, 336), (2033, 2048, 337), (2048, 2048, 351),
                                   (1030, 3000, 400), (1100, 2100, 705), (904, 3244, 1544)])
def test_two_k_groups_on_128_tiles(pkg, dev, m, n, k):
    """One tile to a CU at most: K that ends in either group's slab, with rows and columns of a tile missing, the epilogue
    in the share of the rows that a group finishes, a value that the split cannot represent in each share"""
    import torch
    assert kernel_of(m, n, k) == K128 and -(-m // 128) * -(-n // 128) <= 256
    gen = torch.Generator(device=dev).manual_seed(m + n + k)
    a, b = torch.randn(m, k, device=dev, generator=gen), torch.randn(k, n, device=dev, generator=gen)
    bias = torch.randn(n, device=dev, generator=gen)
    want = a.double() @ b.double()
    out = pkg.blas_matmul(a, b)
    assert rel(out, want) <= bound(k)
    assert torch.equal(pkg.blas_matmul(a, b, bias), out + bias)
    c = torch.full((m, n + 3), float("nan"), device=dev)
    pkg.sgemm_general(a, b.t().contiguous(), c, m, n, k, k, k, n + 3, trans_b=True)
    assert torch.equal(c[:, :n], out) and bool(torch.isnan(c[:, n:]).all())
    a[5, 1], a[m - 1, k - 1] = float("inf"), float("nan")
    got = pkg.blas_matmul(a, b)
    bad = torch.zeros(m, dtype=torch.bool, device=dev)
    bad[5] = bad[m - 1] = True
    assert torch.equal(got[~bad], out[~bad]) and not bool(torch.isfinite(got[bad]).any())


@pytest.mark.parametrize("kernel,m,n,k", ONE_OF_EACH)
def test_every_pair_of_pieces(pkg, dev, kernel, m, n, k):
    """One product to a result, of operands that have all three parts on one side, or the second on both: exact, if no term
    is left out or taken twice."""
    import torch
    assert kernel_of(m, n, k) == kernel
    gen = torch.Generator(device=dev).manual_seed(k)
    full = lambda *s: 1 + torch.randint(0, 1 << 23, s, device=dev, generator=gen).float() * 2.0 ** -23  # noqa: E731
    power = lambda *s: torch.exp2(torch.randint(-9, 9, s, device=dev, generator=gen).float())  # noqa: E731
    second = lambda *s: 1 + 2.0 ** -9 * torch.randint(-1, 2, s, device=dev, generator=gen)  # noqa: E731
    at = (torch.arange(m, device=dev) * 7 + 3) % k
    for left, right in ((full, power), (power, full), (second, second)):
        a = torch.zeros(m, k, device=dev)
        values = left(m)
        a[torch.arange(m, device=dev), at] = values
        b = right(k, n)
        want = (values.double()[:, None] * b.double()[at]).float()
        assert torch.equal(pkg.blas_matmul(a, b), want)
        c = torch.empty(m, n, device=dev)
        pkg.sgemm_general(a, b.t().contiguous(), c, m, n, k, k, k, n, trans_b=True)
        assert torch.equal(c, want)


@pytest.mark.parametrize("share", [0.0, 0.02, 0.1, 0.5, 1.0])
@pytest.mark.parametrize("kernel,m,n,k", ONE_OF_EACH)
def test_sparse_operands_are_summed_no_worse_than_in_fp32(pkg, dev, kernel, m, n, k, share):
    """Rows with a `share` of values that are not zero (0: one of them), against a chain of fp32 multiply-adds over ascending k."""
    import torch
    assert kernel_of(m, n, k) == kernel
    gen = torch.Generator(device=dev).manual_seed(int(share * 100))
    a, b = torch.randn(m, k, device=dev, generator=gen), torch.randn(k, n, device=dev, generator=gen)
    if share == 0:
        at = torch.arange(m, device=dev) % k
        a = torch.zeros_like(a).scatter_(1, at[:, None], a.gather(1, at[:, None]))
    else:
        a *= torch.rand(m, k, device=dev, generator=gen) < share
    rows, cols = slice(0, m, m // 100), slice(0, n, n // 300)
    got, x, y = pkg.blas_matmul(a, b)[rows, cols].double(), a[rows].double(), b[:, cols].double()
    want = x @ y
    if share == 0:
        # half a unit for the sum, 2^-24.2 for the products of pieces that are not formed: below 2^-23 together
        assert bool(((got - want).abs() <= 2.0 ** -23 * want.abs()).all())
        return
    chain = torch.zeros_like(want)
    for i in range(k):
        chain = (chain + x[:, i:i + 1] * y[i:i + 1]).float().double()
    print(rel(got, want), rel(chain, want))
    assert rel(got, want) <= rel(chain, want)


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
    assert rel(out, 0.5 * x * (1 + torch.erf(x / 2 ** 0.5))) <= bound_fp32(k) + 1e-6  # GELU itself: 1e-6


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
    assert rel(out[plain], want[plain]) <= bound_fp32(k) * 2  # tiles with a bad value: fp32 matrix ops, one addition for two k


def test_results_that_cancel(pkg, dev):
    """A few results that are zero among large ones, which the kernel looks at again."""
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
    assert rel(out, a.double() @ b.double() + bias.double()) <= bound_fp32(k)
    # sums of pairs that cancel exactly in any order of fp32 additions that keeps the pairs, and nearly in the others
    assert abs(out[100, 33] - bias[33]) < 1e-4 and abs(out[100, 1999] - bias[1999]) < 1e-4
    a[100] = 0.0
    a[100, 7], a[100, 8] = 1.0, 1.0
    b[7, 40], b[8, 40] = 3.0, -3.0
    out = pkg.blas_matmul(a, b, bias)
    assert out[100, 40] == bias[40]
    assert rel(out, a.double() @ b.double() + bias.double()) <= bound_fp32(k)


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


@pytest.mark.parametrize("kernel,m,n,k", ONE_OF_EACH)
def test_zeros_cost_nothing(pkg, dev, kernel, m, n, k):
    """Padding, a quarter of the rows and a column: 0.97 to 1.01 times the time of the product without (1.4 to 2.0, when a
    tile with a row of zeros read its operands again).  The smaller of twenty times of eight products each."""
    import torch
    assert kernel_of(m, n, k) == kernel
    gen = torch.Generator(device=dev).manual_seed(k)
    a, b = torch.randn(m, k, device=dev, generator=gen), torch.randn(k, n, device=dev, generator=gen)
    x, y = a.clone(), b.clone()
    x[m - m // 4:] = 0
    y[:, 33] = 0
    out = pkg.blas_matmul(x, y)
    assert torch.equal(out[:m - m // 4, :33], pkg.blas_matmul(a, b)[:m - m // 4, :33])
    assert not bool(out[m - m // 4:].any()) and not bool(out[:, 33].any())
    best = [float("inf")] * 2
    for _ in range(20):
        for i, (left, right) in enumerate(((a, b), (x, y))):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(8):
                pkg.blas_matmul(left, right)
            end.record()
            end.synchronize()
            best[i] = min(best[i], start.elapsed_time(end))
    print(kernel, best, best[1] / best[0])
    assert best[1] <= 1.2 * best[0]


@pytest.mark.parametrize("kernel,m,n,k", ONE_OF_EACH)
def test_other_rows_and_columns_do_not_matter(pkg, dev, kernel, m, n, k):
    """A row's results have the same bits whatever its neighbours hold: infinities, NaN, large, tiny and zero ones."""
    import torch
    assert kernel_of(m, n, k) == kernel
    gen = torch.Generator(device=dev).manual_seed(k)
    a, b = torch.randn(m, k, device=dev, generator=gen), torch.randn(k, n, device=dev, generator=gen)
    plain = pkg.blas_matmul(a, b)
    x, y = a.clone(), b.clone()
    x[5, 3], x[40, k - 1], x[77] = float("inf"), float("nan"), 0.0
    x[300], x[333, 7] = a[300] * 2.0 ** -125, 2.0 ** 100
    y[9, 70], y[:, 200] = -float("inf"), b[:, 200] * 2.0 ** 40
    rows = [i for i in range(m) if i not in (5, 40, 77, 300, 333)]
    cols = [j for j in range(n) if j not in (70, 200)]
    out = pkg.blas_matmul(x, y)
    assert torch.equal(out[rows][:, cols], plain[rows][:, cols])
    assert torch.equal(torch.isnan(out), torch.isnan(x.double() @ y.double())) and not bool(out[77][cols].any())
    c = torch.empty(m, n, device=dev)
    pkg.sgemm_general(x, y.t().contiguous(), c, m, n, k, k, k, n, trans_b=True)
    assert torch.equal(c[rows][:, cols], plain[rows][:, cols])
    want = x[300].double() @ y[:, cols].double()
    assert rel(out[300][cols], want) <= bound_fp32(k)


@pytest.mark.parametrize("n", [961, 962, 963])
@pytest.mark.parametrize("row", [70, 1019])
def test_tiny_results_in_the_last_columns_stay_in_their_row(pkg, dev, n, row):
    """One tiny row and one to three columns in the last 64 x 64 tiles: few results to look at again, next to the columns that a
    load of four has beyond N.  The next row, the columns behind N of a wider result, and what lies behind the last row stay."""
    import torch
    m, k = 1020, 2050
    assert kernel_of(m, n, k) == K64
    gen = torch.Generator(device=dev).manual_seed(n + row)
    a, b = torch.randn(m, k, device=dev, generator=gen), torch.randn(k, n, device=dev, generator=gen)
    plain = pkg.blas_matmul(a, b)
    a[row] *= 2.0 ** -80
    rest = [i for i in range(m) if i != row]
    for ldc in (n, n + 5):
        c = torch.full((m * ldc + 8,), 7.0, device=dev)
        pkg.sgemm_general(a, b, c, m, n, k, k, n, ldc)
        out = c[:m * ldc].view(m, ldc)
        assert torch.equal(out[rest, :n], plain[rest]) and bool((c[m * ldc:] == 7).all()) and bool((out[:, n:] == 7).all())
        assert rel(out[row, :n], a[row].double() @ b.double()) <= bound_fp32(k)


@pytest.mark.parametrize("kernel,m,n,k", [(WIDE, 3969, 3841, 600), (K128, 2047, 1921, 1009), (K64, 1020, 962, 2050)])
def test_tiny_results_have_the_bits_of_large_ones(pkg, dev, kernel, m, n, k):
    """Rows scaled by 2^-75, one of them or many together, in tiles that are full and in the last ones, of one or two columns: the
    results are those of the rows as they were, scaled, however many of a tile's are small."""
    import torch
    assert kernel_of(m, n, k) == kernel
    gen = torch.Generator(device=dev).manual_seed(m)
    a, b = torch.randn(m, k, device=dev, generator=gen), torch.randn(k, n, device=dev, generator=gen)
    bt = b.t().contiguous()
    plain = pkg.blas_matmul(a, b)
    for rows in ([70], list(range(64, 128))):
        x, want = a.clone(), plain.clone()
        x[rows] *= 2.0 ** -75
        want[rows] *= 2.0 ** -75
        assert torch.equal(pkg.blas_matmul(x, b), want)
        c = torch.empty(m, n, device=dev)
        pkg.sgemm_general(x, bt, c, m, n, k, k, k, n, trans_b=True)
        assert torch.equal(c, want)


# a batch of each: true batches, every entry with its own operands
BATCHED = [(WIDE, 1021, 1030, 769, 6), (K128, 650, 770, 515, 12), (K64, 251, 510, 1565, 8)]


@pytest.mark.parametrize("kernel,m,n,k,batch", BATCHED + [(kind, m, n, k, 1) for kind, m, n, k in ONE_OF_EACH])
def test_fused_epilogues_have_the_bits_of_separate_steps(pkg, dev, kernel, m, n, k, batch):
    import torch
    assert kernel_of(m, n, k, batch) == kernel
    gen = torch.Generator(device=dev).manual_seed(m)
    a, b, r = (torch.randn(*s, device=dev, generator=gen) for s in ((batch, m, k), (batch, k, n), (batch, m, n)))
    bias = torch.randn(n, device=dev, generator=gen)
    plain = pkg.blas_matmul(a, b)
    for act in (0, 1):
        out = torch.empty(batch, m, n, device=dev)
        pkg.check(pkg.lib().tfcc_rocm_sgemm_fused(None, a.data_ptr(), m * k, b.data_ptr(), k * n, bias.data_ptr(), r.data_ptr(),
                                                  m * n, out.data_ptr(), m * n, m, n, k, batch, act))
        want = plain + bias + r
        assert torch.equal(out, pkg.gelu_accurate(want) if act else want)


@pytest.mark.parametrize("kernel,m,n,k", ONE_OF_EACH)
def test_products_that_share_a_have_the_bits_of_single_ones(pkg, dev, kernel, m, n, k):
    import torch
    assert kernel_of(m, n, k) == kernel
    gen = torch.Generator(device=dev).manual_seed(n)
    a = torch.randn(m, k, device=dev, generator=gen)
    a[m - 1] *= 2.0 ** -120  # formed again with the fp32 matrix ops
    for groups in (2, 4):
        bs = [torch.randn(k * n + g, device=dev, generator=gen)[g:].view(k, n) for g in range(groups)]
        biases = [torch.randn(n, device=dev, generator=gen) for _ in bs]
        for got, b, bias in zip(pkg.sgemm_grouped(a, bs, biases), bs, biases):
            assert torch.equal(got, pkg.blas_matmul(a, b, bias))


@pytest.mark.parametrize("kernel,m,n,k,batch", BATCHED)
def test_batches_of_padded_matrices_with_special_values_in_each(pkg, dev, kernel, m, n, k, batch):
    """Two-level batches, rows with padding behind them, and in every entry other rows that have to be formed again (for which
    the operands are read from where the entry's lie), with bias and GELU on top; B as stored and transposed."""
    import torch
    assert kernel_of(m, n, k, batch) == kernel
    gen = torch.Generator(device=dev).manual_seed(k)
    lda, ldb, ldt, ldc = k + 3, n + 1, k + 2, n + 5
    a, b = torch.randn(batch, m, lda, device=dev, generator=gen), torch.randn(batch, k, ldb, device=dev, generator=gen)
    bias = torch.randn(n, device=dev, generator=gen)
    for i in range(batch):
        a[i, 3 * i + 1, 7 * i] = float("inf")
        a[i, 64 + i, :k] *= 2.0 ** -120
        a[i, 140 + i, :k] = 0.0
        a[i, 140 + i, 5 + i] = 2.0 ** -135
        b[i, 5 + i, :n] = 2.0 ** 110
        a[i, :140 + i, 5 + i] = 0.0
        a[i, 141 + i:, 5 + i] = 0.0
    bt = torch.zeros(batch, n, ldt, device=dev)
    bt[:, :, :k] = b[:, :, :n].transpose(1, 2)
    outer, inner = batch // 2, 2
    x, y = a[:, :, :k], b[:, :, :n]
    want = torch.stack([x[i].double() @ y[i].double() for i in range(batch)]) + bias.double()
    outs = []
    for tb, act in ((False, 0), (True, 0), (False, 1), (True, 1)):
        c = torch.full((batch, m, ldc), 7.0, device=dev)
        right, ld, size = (bt, ldt, n * ldt) if tb else (b, ldb, k * ldb)
        pkg.sgemm_general(a, right, c, m, n, k, lda, ld, ldc, trans_b=tb, batch_outer=outer, batch_inner=inner,
                          strides=(2 * m * lda, 2 * size, 2 * m * ldc), inner_strides=(m * lda, size, m * ldc), bias=bias, activation=act)
        assert bool((c[:, :, n:] == 7).all())
        outs.append(c[:, :, :n].contiguous())
    assert torch.equal(outs[0].nan_to_num(), outs[1].nan_to_num()) and torch.equal(outs[2].nan_to_num(), outs[3].nan_to_num())
    assert torch.equal(outs[2].nan_to_num(), pkg.gelu_accurate(outs[0]).nan_to_num())
    finite = torch.isfinite(want)
    assert torch.equal(torch.isfinite(outs[0]), finite)
    for i in range(batch):
        assert torch.equal(outs[0][i, 140 + i], (bias.double() + 2.0 ** -25).float())
        rows = [j for j in range(m) if j != 3 * i + 1]
        assert rel(outs[0][i, rows], want[i, rows]) <= bound_fp32(k)


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("kernel,m,n,k", [(WIDE, 3969, 3841, 600), (K128, 2047, 1921, 1009), (K64, 1020, 962, 2050)])
def test_a_few_results_that_the_split_gets_wrong(pkg, dev, kernel, m, n, k, trans_b):
    """Single results that are small next to a small operand, fewer than a tile lists, in full tiles and in the last ones: as the
    fp32 matrix ops have them, bias and GELU on top, and nothing else is touched."""
    import torch
    assert kernel_of(m, n, k) == kernel
    gen = torch.Generator(device=dev).manual_seed(m)
    a, b = torch.randn(m, k, device=dev, generator=gen), torch.randn(k, n, device=dev, generator=gen)
    a[:, 9] = 0.0
    plain = product(pkg, a, b, trans_b)
    row, cols = 70, [3, 40, 500, n - 1]
    a[row] = 0.0
    a[row, 9] = 1.2345678 * 2.0 ** -115  # the third part of it lies outside bf16's range
    b[9] = 0.0
    b[9, cols] = torch.tensor([1.0, -1.5, 3.0, 0.5], device=dev)
    want = torch.zeros(n, dtype=torch.double, device=dev)
    want[cols] = a[row, 9].double() * b[9, cols].double()
    out = product(pkg, a, b, trans_b)
    assert torch.equal(out[row].double(), want.float().double())
    rest = [i for i in range(m) if i != row]
    assert torch.equal(out[rest], plain[rest])


def product(pkg, a, b, trans_b):
    import torch
    (m, k), n = a.shape, b.shape[1]
    if not trans_b:
        return pkg.blas_matmul(a, b)
    return pkg.sgemm_general(a, b.t().contiguous(), torch.empty(m, n, device=a.device), m, n, k, k, k, n, trans_b=True)
