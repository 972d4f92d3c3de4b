"""Dense Q8_0 products of large batches (q8_wide_k, k_gemm.hip) against the CPU oracle: the three widths of a block, rows and tokens
that do not fill the last one, row counts that are no multiple of four, two to 32 stages.  Exact mode keeps the oracle's bits; fast mode
fuses the scaled add: at most 128 roundings of 2^-24 of sums no larger than a few times the row's largest result."""
import numpy as np
import pytest

from util import q8_0_weights, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("n_in,n_out,n", [
    (256, 4097, 400), (512, 8190, 209), (1280, 4224, 385), (4096, 2050, 899),        # 32 tokens a block
    (256, 8062, 500), (768, 8191, 450), (2048, 1030, 4033),                           # 64
    (256, 8130, 1481), (512, 8065, 1409), (2048, 4100, 2049), (4096, 1025, 8191),     # 128
])
def test_wide_tiles(exact, n_in, n_out, n):
    import inferred_hip as ih
    from oracle import binding as ob
    orc = ob.Oracle(threads=8)
    be = ih.Hip(exact=exact)
    try:
        r = rng(n_in + n_out + n)
        w = q8_0_weights(orc, r, n_out, n_in, std=0.05)
        x = (r.standard_normal((n, n_in), dtype=np.float32) * 10.0 ** r.uniform(-2, 2, (n, 1)).astype(np.float32)).reshape(-1)
        a = np.full(n * n_out, np.nan, np.float32)
        be.matmul(ih.weights(w, ih.Q8_0, n_in, n_out), x, a)
        be.host_needs(a)
        be.raise_if_error()
        got = a.reshape(n, n_out)
        assert np.isfinite(got).all()
        rows = np.unique(np.r_[0:3, 31:34, n // 2 - 2:n // 2 + 2, n - 34:n])          # the oracle on the edges of the tiles
        xs = np.ascontiguousarray(x.reshape(n, n_in)[rows]).reshape(-1)
        b = np.zeros(len(rows) * n_out, np.float32)
        orc.matmul(ob.weights(w, ih.Q8_0, n_in, n_out), xs, b)
        got, want = got[rows], b.reshape(len(rows), n_out)
        if exact:
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        else:
            assert (np.abs(got - want).max(1) <= 1e-5 * np.abs(want).max(1)).all()
    finally:
        be.close()
