"""Quantized products of at most one 64 x 128 tile for each CU and more than 768 k, whose slabs pass through a ring of four
stages: from 70 tiles to the last size that takes them (256), a last slab of 16 k, ragged rows and columns, batches; bit for bit
against the oracle, with the int32 result, the requantized one and both."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

# m, k, n, batch: 65 to 256 tiles, K just above 768, whole slabs of 128 and all remainders' ends
SHAPES = [(1024, 784, 2048, 1), (833, 896, 640, 1), (1025, 1008, 1920, 1), (4096, 912, 512, 1), (65, 2064, 4240, 1),
          (300, 1024, 656, 3), (333, 4112, 2064, 1)]


@pytest.mark.parametrize("m,k,n,batch", SHAPES)
def test_against_the_oracle(pkg, T, m, k, n, batch):
    tiles = -(-m // 64) * -(-n // 128) * batch
    assert 64 < tiles <= 256 and k > 768 and k % 16 == 0 and n % 16 == 0
    rng = np.random.default_rng(m + 3 * k + n)
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
    ta, tb, trs, tcs = T.t(a), T.t(b), T.t(rs), T.t(cs)
    for exact in (False, True):
        for acc_wanted in (False, True):
            q, acc, _, _ = pkg.quantization_matmul_requantize(ta, trs, r[0], r[1], tb, tcs, r[2], r[3], T.f1(lo), T.f1(hi),
                                                              want_acc=acc_wanted, colsum_exact=exact)
            assert np.array_equal(T.n(q), want_q)
            assert not acc_wanted or np.array_equal(T.n(acc), want)
    c, _, _ = pkg.quantization_matmul(ta, trs, r[0], r[1], tb, tcs, r[2], r[3])
    assert np.array_equal(T.n(c), want)
