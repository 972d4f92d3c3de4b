"""Dense Q8_0 products of short batches in fast mode (k_q8_short.hip) against the CPU oracle: every row length the kernel takes
(256 k per wave, one to eight waves, twice that at 4,096), ragged row and token counts, both row heights of a block, and sizes
just outside its rule, which take the tiles or the GEMVs.  The int32 block sums are the oracle's; the f32 sums run in another
order: |error| <= 1e-5 of the row's largest result."""
import numpy as np
import pytest

from util import q8_0_weights, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_in,n_out,n", [(256, 8192, 2), (256, 100, 16), (512, 33, 17), (512, 4096, 33), (1024, 66, 64), (1024, 510, 200),
                                          (2048, 512, 31), (2048, 4099, 5), (2048, 8192, 32), (2048, 8192, 33), (4096, 2048, 23),
                                          (4096, 130, 128), (4096, 2048, 129), (1536, 64, 20), (2048, 512, 15)])
def test_short_batches(n_in, n_out, n):
    import inferred_hip as ih
    from oracle import binding as ob
    orc = ob.Oracle(threads=8)
    be = ih.Hip(exact=False)
    try:
        r = rng(n_in + n_out + n)
        w = q8_0_weights(orc, r, n_out, n_in, std=0.05)
        x = (r.standard_normal(n * n_in) * np.repeat(10.0 ** r.uniform(-2, 2, n), n_in)).astype(np.float32)
        a, b = np.zeros(n * n_out, np.float32), np.zeros(n * n_out, np.float32)
        be.matmul(ih.weights(w, ih.Q8_0, n_in, n_out), x, a)
        be.host_needs(a)
        be.raise_if_error()
        orc.matmul(ob.weights(w, ih.Q8_0, n_in, n_out), x, b)
        for t in range(n):
            s = slice(t * n_out, (t + 1) * n_out)
            assert np.abs(a[s] - b[s]).max() <= 1e-5 * np.abs(b[s]).max(), (t, np.abs(a[s] - b[s]).max(), np.abs(b[s]).max())
    finally:
        be.close()


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("n_in,n_out,n", [(256, 64, 33), (512, 130, 40), (2048, 8192, 70), (2048, 8192, 100), (2048, 514, 1300),
                                          (4096, 2046, 65), (256, 8192, 4200), (2048, 66, 17)])
def test_tiles_over_whole_slabs(exact, n_in, n_out, n):
    """q8_tile_k (k_gemm.hip): one to sixteen stages, the three token widths of a block with ragged ends; exact mode keeps the
    oracle's bits."""
    import inferred_hip as ih
    from oracle import binding as ob
    orc = ob.Oracle(threads=8)
    be = ih.Hip(exact=exact)
    try:
        r = rng(n_in + n_out + n)
        w = q8_0_weights(orc, r, n_out, n_in, std=0.05)
        x = (r.standard_normal(n * n_in) * np.repeat(10.0 ** r.uniform(-2, 2, n), n_in)).astype(np.float32)
        a = np.zeros(n * n_out, np.float32)
        be.matmul(ih.weights(w, ih.Q8_0, n_in, n_out), x, a)
        be.host_needs(a)
        be.raise_if_error()
        rows = np.unique(np.r_[0:3, n // 2, n - 18:n])          # the oracle on the edges of the tiles
        xs = np.ascontiguousarray(x.reshape(n, n_in)[rows]).reshape(-1)
        b = np.zeros(len(rows) * n_out, np.float32)
        orc.matmul(ob.weights(w, ih.Q8_0, n_in, n_out), xs, b)
        got, want = a.reshape(n, n_out)[rows], b.reshape(len(rows), n_out)
        if exact:
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        else:
            assert (np.abs(got - want).max(1) <= 1e-5 * np.abs(want).max(1)).all()
    finally:
        be.close()
