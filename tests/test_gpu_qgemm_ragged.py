"""Quantized products of every size class and alignment of the dispatch against the oracle, bit for bit: the kernel without
slabs in each of its tiles, the one for operands shorter than a load, the slab kernels with one and two K groups, and the
skinny product with per-channel dequantize on shapes that the streaming kernels do not take."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

# m, k, n, batch
SHAPES = [
    (1, 1, 1, 1), (3, 5, 2, 1), (1, 15, 40, 1), (5, 3, 1, 2), (1, 1, 5000, 1), (7, 2, 1, 1), (15, 1, 3, 3),   # shorter than a load
    (1, 16, 1, 1), (2, 8, 7, 1), (16, 17, 65, 1), (17, 63, 63, 1), (15, 64, 130, 1), (33, 65, 61, 2),           # 16 rows, one step of k
    (9, 449, 67, 1), (77, 1001, 1237, 1), (16, 2047, 130, 1), (20, 4099, 71, 1), (8, 3999, 700, 1),             # 8 and 16 wavefronts
    (128, 769, 3070, 1), (33, 385, 4095, 1), (90, 401, 500, 5), (65, 300, 1000, 2),                              # 32 rows
    (450, 2050, 1023, 1), (129, 4003, 640, 1),                                                                   # 64 rows
    (513, 1023, 1025, 1), (1000, 500, 2001, 1), (515, 257, 1030, 1), (100, 300, 200, 40),                        # 64 x 128, two K groups
    (1344, 959, 1948, 1), (2000, 400, 1999, 1),                                                                  # 128 x 128, two K groups
    (2000, 64, 2001, 1), (3000, 200, 3001, 1), (130, 100, 131, 70), (3584, 130, 3585, 1),                        # one K group
    (4, 65, 1, 1), (16, 66, 1, 1), (9, 67, 1, 1), (40, 129, 1, 1), (300, 130, 1, 1), (2049, 193, 1, 1), (5, 257, 1, 1),  # one column
    (3, 65, 2, 1), (7, 66, 3, 1), (33, 130, 2, 3), (4000, 65, 1, 1), (40, 130, 1, 40), (8, 4097, 1, 1),
    (5000, 129, 1, 1), (5000, 258, 1, 1), (40, 130, 1, 70), (33000, 385, 1, 1), (5000, 131, 1, 1), (5000, 130, 3, 1),  # in slabs
    (100000, 129, 1, 1), (40, 257, 2, 800),
    (256, 1024, 1024, 1), (32, 512, 4096, 1), (64, 64, 64, 6), (520, 512, 1024, 1),                              # aligned, both sides of the line
]


def _unaligned(torch, x, by):
    flat = torch.empty(x.numel() + by, dtype=x.dtype, device="cuda")
    flat[by:].copy_(x.reshape(-1))
    return flat[by:].view(x.shape)


@pytest.mark.parametrize("m,k,n,batch", SHAPES)
def test_ragged_quantized_products(pkg, T, m, k, n, batch):
    import torch
    print("qgemm ragged", m, k, n, batch, flush=True)
    rng = np.random.default_rng(m * 11 + k * 5 + n)
    lead = () if batch == 1 else (batch,)
    a = rng.integers(0, 256, lead + (m, k), dtype=np.uint8)
    b = rng.integers(-128, 128, lead + (k, n), dtype=np.int8)
    rs, cs = O.reduce_sum(a, True), O.reduce_sum(b, False)
    ranges = (-100.0, 155.0, -117.0, 138.0)
    oa, ob = O.qmatmul_offsets(*ranges)
    want = O.qgemm(a, b, oa, ob, rs, cs)
    mn_c, mx_c = O.qmatmul_range(*ranges)
    real = O.dequantize(want, mn_c, mx_c).astype(np.float64)
    lo = float(np.float32(real.min() + 0.1 * (np.ptp(real) + 1)))
    hi = float(np.float32(real.max() + 1))
    want_q = O.requantize_s32_u8(want, mn_c, mx_c, lo, hi)
    r = [T.f1(v) for v in ranges]
    for shift in (0, 1, 3):
        ta, tb = _unaligned(torch, T.t(a), shift), _unaligned(torch, T.t(b), shift)
        c, got_lo, got_hi = pkg.quantization_matmul(ta, T.t(rs), r[0], r[1], tb, T.t(cs), r[2], r[3])
        assert np.array_equal(T.n(c), want), shift
        assert (float(T.n(got_lo)[0]), float(T.n(got_hi)[0])) == (mn_c, mx_c)
        for exact in (False, True):
            q, acc, _, _ = pkg.quantization_matmul_requantize(ta, T.t(rs), r[0], r[1], tb, T.t(cs), r[2], r[3], T.f1(lo), T.f1(hi),
                                                              want_acc=exact, colsum_exact=exact)
            assert np.array_equal(T.n(q), want_q), (shift, exact)
            assert acc is None or np.array_equal(T.n(acc), want)


@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (2, 7, 5), (8, 2153, 897), (3, 1001, 12), (5, 64, 66), (7, 4095, 130), (8, 700, 3001),
                                   (1, 65, 1), (4, 66, 1), (8, 129, 1), (3, 1025, 1), (2, 4098, 1), (5, 67, 1), (6, 130, 2)])
def test_ragged_skinny_product_dequantized(pkg, T, m, k, n):
    rng = np.random.default_rng(m + k + n)
    a = rng.integers(0, 256, (m, k), dtype=np.uint8)
    b = rng.integers(-127, 128, (k, n), dtype=np.int8)
    scale = rng.uniform(0.001, 0.01, n).astype(np.float32)
    rs, cs = O.reduce_sum(a, True), O.reduce_sum(b, False)
    want = O.qgemm(a, b, -57, 93, rs, cs)
    want_f = (want.astype(np.float64) * (np.float64(np.float32(0.02)) * scale.astype(np.float64))).astype(np.float32)
    for exact in (False, True):
        for keep in (False, True):
            out, acc = pkg.gemv_dequant(T.t(a), T.t(b), T.t(rs), T.t(cs), -57, 93, 0.02, T.t(scale), want_acc=keep, colsum_exact=exact)
            assert np.array_equal(T.n(out).view(np.uint32), want_f.view(np.uint32))
            assert (acc is not None) == keep and (acc is None or np.array_equal(T.n(acc), want))
