"""Quantized products in slabs whose rows and addresses are multiples of four bytes but not of sixteen (copies, with stores of
their own) or of nothing (registers), on both tile heights and with one and two slabs on their way: bit for bit against the oracle."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

# m, k, n, batch, bytes by which the operands are moved
SHAPES = [
    (600, 772, 836, 1, 0), (641, 896, 1004, 1, 4), (4100, 900, 132, 1, 8), (65, 1028, 8452, 1, 0),       # words, four stages
    (1030, 4, 1028, 1, 0), (1700, 132, 1284, 1, 12), (700, 260, 3972, 1, 4), (130, 20, 260, 40, 4),     # words, 64 rows
    (2100, 1668, 2052, 1, 0), (2309, 516, 3588, 1, 4),                                                  # words, 128 rows
    (640, 1024, 1024, 1, 4), (2048, 128, 1040, 1, 2),                                                   # round sizes at other addresses
    (600, 769, 835, 1, 0), (641, 897, 1003, 1, 1), (513, 1025, 1031, 1, 3), (4100, 1153, 130, 1, 0),     # bytes, two slabs under way
    (1030, 5, 1029, 1, 0), (70000, 4, 4, 1, 0), (70000, 3, 5, 1, 0), (2100, 1670, 2051, 1, 1),           # bytes: short K, 128 rows
]


def _moved(torch, x, by):
    flat = torch.empty(x.numel() + by, dtype=x.dtype, device="cuda")
    flat[by:].copy_(x.reshape(-1))
    return flat[by:].view(x.shape)


@pytest.mark.parametrize("m,k,n,batch,by", SHAPES)
def test_products_in_slabs_at_any_address(pkg, T, m, k, n, batch, by):
    import torch
    print("qgemm words", m, k, n, batch, by, flush=True)
    rng = np.random.default_rng(m * 7 + k * 3 + n)
    lead = () if batch == 1 else (batch,)
    a = rng.integers(0, 256, lead + (m, k), dtype=np.uint8)
    b = rng.integers(-128, 128, lead + (k, n), dtype=np.int8)
    rs, cs = O.reduce_sum(a, True), O.reduce_sum(b, False)
    ranges = (-100.0, 155.0, -117.0, 138.0)
    want = O.qgemm(a, b, *O.qmatmul_offsets(*ranges), rs, cs)
    mn_c, mx_c = O.qmatmul_range(*ranges)
    real = O.dequantize(want, mn_c, mx_c).astype(np.float64)
    lo, hi = float(np.float32(real.min() + 0.1 * np.ptp(real))), float(np.float32(real.max() + 1))
    want_q = O.requantize_s32_u8(want, mn_c, mx_c, lo, hi)
    r = [T.f1(v) for v in ranges]
    ta, tb = _moved(torch, T.t(a), by), _moved(torch, T.t(b), by)
    c, _, _ = pkg.quantization_matmul(ta, T.t(rs), r[0], r[1], tb, T.t(cs), r[2], r[3])
    assert np.array_equal(T.n(c), want)
    for both in (False, True):
        q, acc, _, _ = pkg.quantization_matmul_requantize(ta, T.t(rs), r[0], r[1], tb, T.t(cs), r[2], r[3], T.f1(lo), T.f1(hi),
                                                          want_acc=both, colsum_exact=both)
        assert np.array_equal(T.n(q), want_q), both
        assert acc is None or np.array_equal(T.n(acc), want)
