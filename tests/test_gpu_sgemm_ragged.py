"""fp32 products whose K ends inside a slab of 32, whose rows are no multiple of four long or whose operands are not aligned
to 16 bytes: on every kernel of the dispatch, against float64, and with rows of A that are not finite between the others (what
lies past the end of a row is the next one, and must not be multiplied)."""
import numpy as np
import pytest

from conftest import rel_fro

pytestmark = pytest.mark.gpu

# m, k, n, batch: one line per kernel the dispatcher picks (32x32, 32x64, 32x96 and 64x64 tiles with one, two and four K
# groups; 128 x 96 and 128 x 128 tiles), each with K just past and just before a slab's end and n % 4 of 1, 2 and 3
SHAPES = [(9, 1, 1, 1), (33, 31, 66, 1), (64, 33, 65, 1), (31, 97, 31, 1), (100, 63, 97, 1),
          (40, 257, 33, 1), (65, 287, 130, 1), (200, 319, 333, 1), (400, 289, 399, 1), (640, 300, 1021, 1),
          (33, 513, 97, 1), (77, 1001, 1237, 1), (333, 1003, 517, 1), (128, 767, 3071, 1), (129, 770, 3074, 1), (700, 1025, 1023, 1), (960, 2047, 1022, 1),
          (1021, 513, 3071, 1), (2047, 515, 2046, 1), (2045, 67, 4090, 1), (33, 64, 65, 1), (128, 96, 131, 1), (512, 512, 514, 1),
          (29, 29, 64, 12), (29, 64, 29, 12), (50, 45, 51, 7), (130, 61, 127, 192), (65, 300, 63, 40)]


@pytest.mark.parametrize("m,k,n,batch", SHAPES)
def test_ragged_products(pkg, T, m, k, n, batch):
    import torch
    print("ragged", m, k, n, batch, flush=True)
    rng = np.random.default_rng(m * 7 + k * 3 + n)
    a = rng.standard_normal((batch, m, k), dtype=np.float32)
    b = rng.standard_normal((batch, k, n), dtype=np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    a[:, 1::2] = np.inf
    shape = (lambda x: x[0]) if batch == 1 else (lambda x: x)
    got = T.n(pkg.blas_matmul(T.t(shape(a)), T.t(shape(b)), T.t(bias))).reshape(batch, m, n)
    want = np.matmul(a[:, ::2].astype(np.float64), b.astype(np.float64)) + bias
    # sums of K products in fp32: relative error of the norm below sqrt(K) 2^-24 < 3e-6 at the largest K here
    assert rel_fro(got[:, ::2], want) <= 5e-6
    # the same from operands that start four bytes past an aligned address
    pad = lambda x: torch.cat([torch.zeros(1, device="cuda"), T.t(x).reshape(-1)])[1:].view(x.shape)
    off = T.n(pkg.blas_matmul(pad(shape(a)), pad(shape(b)), T.t(bias))).reshape(batch, m, n)
    assert np.array_equal(off[:, ::2], got[:, ::2])
    # B handed over transposed is summed in the same order
    if batch == 1 and m > 8:
        out = torch.empty((m, n), device="cuda")
        pkg.sgemm_general(T.t(a[0]), T.t(b[0].T.copy()), out, m, n, k, k, k, n, trans_b=True, bias=T.t(bias))
        assert np.array_equal(T.n(out)[::2], got[0, ::2])
