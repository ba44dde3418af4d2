"""The two ends of a range share an allocation: each is a tensor of one element whatever becomes of the other, and one of them is as good
an argument as a tensor by itself."""
import copy

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_ends_of_a_range_are_tensors_of_their_own(pkg, T):
    import torch
    rng = np.random.default_rng(5)
    x, w = T.t(rng.normal(0, 1, (5, 70)).astype(np.float32)), T.t(rng.integers(-127, 128, (70, 9)).astype(np.int8))
    q, low, high = pkg.quantize(x, torch.uint8)
    assert float(low) == float(x.min()) and float(high) == float(x.max())
    for t in (low, high):
        assert t.shape == (1,) and t.stride() == (1,) and t.is_contiguous() and t.dtype == torch.float32 and not t.requires_grad
    row, col = pkg.reduce_sum(q, True), pkg.reduce_sum(w, False)
    low_w, high_w, low_o, high_o = (T.f1(v) for v in (-1.0, 1.0, -9.0, 9.0))
    calls = (lambda lo, hi: pkg.quantization_matmul(q, row, lo, hi, w, col, low_w, high_w),
             lambda lo, hi: pkg.quantization_matmul_requantize(q, row, lo, hi, w, col, low_w, high_w, low_o, high_o)[::2] + (None,))
    for call in calls:
        shared, apart = call(low, high), call(T.f1(float(low)), T.f1(float(high)))
        for a, b in zip(shared, apart):
            assert a is None or torch.equal(a, b)
    c, low_c, high_c = calls[0](low, high)
    before = float(high_c)
    want = pkg.dequantize(c, low_c, high_c)
    assert torch.equal(pkg.dequantize(c, low_c.clone(), high_c.clone()), want)
    kept, twin = float(low_c), copy.deepcopy(high_c)
    low_c.add_(1000.0)
    assert float(high_c) == before == float(twin) and float(low_c) == np.float32(kept) + np.float32(1000)
    del low_c
    junk = [torch.full((1,), -3.0, device="cuda") for _ in range(64)]
    torch.cuda.synchronize()
    assert float(high_c) == before and len(junk) == 64
