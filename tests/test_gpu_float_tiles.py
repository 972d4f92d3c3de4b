"""Unquantized matrices over a batch in fast mode: the tiles of 16 x 16 to 48 x 64 that the rule gives these sizes, rows and tokens
that do not fill the last one, two matrices of a launch.  Products and sums in f32, in any order: n_in roundings of 2^-24 of the sum
of the products' magnitudes bound the error."""
import numpy as np
import pytest

from util import rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_in", [16, 272, 2048])
@pytest.mark.parametrize("n_a,n_b,n", [
    (512, 1, 64), (33, 31, 3),          # 16 x 16
    (512, 1, 201), (100, 3, 515),       # 16 x 32
    (513, 2, 333), (95, 64, 1001),      # 32 x 32
    (512, 1, 512), (33, 30, 5701), (128, 1, 5700),   # 32 x 64, of eight waves and of four
    (512, 1, 1024), (47, 50, 2049),     # 48 x 48
    (512, 1, 3001), (145, 100, 4097),   # 48 x 64
])
def test_float_tiles(n_in, n_a, n_b, n):
    import inferred_hip as ih
    r = rng(n_in + n)
    wa, wb = r.standard_normal((n_a, n_in), dtype=np.float32), r.standard_normal((n_b, n_in), dtype=np.float32)
    x = r.standard_normal((n, n_in), dtype=np.float32)
    be = ih.Hip(exact=False)
    try:
        a, b = np.full(n * n_a, np.nan, np.float32), np.full(n * n_b, np.nan, np.float32)
        be.matmul_pair(ih.weights(wa.reshape(-1).view(np.uint8), ih.F32, n_in, n_a), ih.weights(wb.reshape(-1).view(np.uint8), ih.F32, n_in, n_b),
                       x.reshape(-1), a, b)
        be.host_needs(a); be.host_needs(b)
        be.raise_if_error()
        for got, w in ((a.reshape(n, n_a), wa), (b.reshape(n, n_b), wb)):
            want = x.astype(np.float64) @ w.astype(np.float64).T
            bound = (n_in + 1) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T)
            assert np.all(np.abs(got - want) <= bound)
    finally:
        be.close()
