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


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("n_in,n_out,n", [(256, 4097, 400), (256, 8062, 500), (256, 8130, 1481)])      # 32, 64, 128 tokens a block
def test_scales_at_the_ends_of_f16(exact, n_in, n_out, n):
    """The scales' products come from f16 operands of the matrix cores: rows and tokens of subnormal steps only (2^-24 and up), with
    zeros among others, and up to the largest finite one."""
    import inferred_hip as ih
    from oracle import binding as ob
    orc = ob.Oracle(threads=8)
    be = ih.Hip(exact=exact)
    try:
        r = rng(n_in + n_out + n)
        nb = n_in // 32

        def steps(rows):
            """f16 steps [rows][nb], five kinds of row in turn"""
            sub = r.integers(1, 1024, (rows, nb)) * 2.0 ** -24
            normal = 10.0 ** r.uniform(-3, 0, (rows, nb))
            kind = (np.arange(rows) % 5)[:, None]
            some = r.random((rows, nb)) < 0.5
            d = np.select([kind == 0, kind == 1, kind == 2, kind == 3], [sub, np.where(some, 0.0, normal), np.where(some, 65504.0, normal),
                                                                         np.where(some, sub, normal)], normal)
            d[0], d[-1] = 2.0 ** -24, 65504.0
            return d.astype(np.float16)

        w = q8_0_weights(orc, r, n_out, n_in, std=0.05).reshape(n_out, nb, 34)
        w[:, :, :2] = steps(n_out)[:, :, None].view(np.uint8)
        w = np.ascontiguousarray(w).reshape(-1)
        q = r.integers(-127, 128, (n, nb, 32)).astype(np.float32)
        q[:, :, 0] = 127                                                   # (the block's step is its largest value / 127)
        x = (q * steps(n).astype(np.float32)[:, :, None]).reshape(-1)
        a = np.full(n * n_out, np.nan, np.float32)
        be.matmul(ih.weights(w, ih.Q8_0, n_in, n_out), x, a)
        be.host_needs(a)
        be.raise_if_error()
        rows = np.unique(np.r_[0:6, 30:36, n // 2 - 2:n // 2 + 2, n - 34:n])
        xs = np.ascontiguousarray(x.reshape(n, n_in)[rows]).reshape(-1)
        b = np.zeros(len(rows) * n_out, np.float32)
        orc.matmul(ob.weights(w, ih.Q8_0, n_in, n_out), xs, b)
        got, want = a.reshape(n, n_out)[rows], b.reshape(len(rows), n_out)
        assert np.isfinite(want).all() and (want[0, ::5] != 0).all()       # (subnormal steps on both sides: nothing larger beside them)
        if exact:
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        else:
            assert (np.abs(got - want).max(1) <= 1e-5 * np.abs(want).max(1)).all()
    finally:
        be.close()
