"""Unquantized matrices over 1 to 300 tokens: the exact mode's fold bit for bit, the fast mode's sums to 1e-5 of the row's scale."""
import numpy as np
import pytest

import inferred_hip as ih

pytestmark = pytest.mark.gpu


def serial(w, x):
    """The CPU path's fold (product and sum each rounded to f32, k ascending), every output at once."""
    s = np.zeros((x.shape[0], w.shape[0]), np.float32)
    for k in range(w.shape[1]):
        s = s + x[:, k:k + 1] * w[None, :, k]
    return s


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("n_in,n0,n1", [(2048, 512, 1), (2048, 32, 32), (4112, 17, 3), (36, 70, 0), (33, 5, 2), (16, 1, 0)])
def test_against_the_serial_fold(exact, n_in, n0, n1):
    r = np.random.default_rng(n_in + n0)
    be = ih.Hip(exact=exact)
    try:
        wa, wb = (r.standard_normal((n, n_in)).astype(np.float32) for n in (n0, max(n1, 1)))
        a, b = ih.weights(wa, ih.F32, n_in, n0), ih.weights(wb, ih.F32, n_in, max(n1, 1))
        for n in (1, 2, 8, 9, 16, 17, 33, 65, 300):
            x = r.standard_normal((n, n_in)).astype(np.float32)
            oa, ob = np.zeros((n, n0), np.float32), np.zeros((n, max(n1, 1)), np.float32)
            be.host_wrote(x)
            if n1:
                be.matmul_pair(a, b, x.reshape(-1), oa.reshape(-1), ob.reshape(-1))
            else:
                be.matmul(a, x.reshape(-1), oa.reshape(-1))
            for got, w in ((oa, wa),) + (((ob, wb),) if n1 else ()):
                be.host_needs(got.reshape(-1))
                want = serial(w, x)
                if exact:
                    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (n, n_in)
                else:
                    assert np.abs(got - want).max() <= 1e-5 * np.sqrt(n_in) * np.abs(x).max(), (n, n_in)
            be.raise_if_error()
            for t in (x, oa, ob):
                be.release(t)
    finally:
        be.close()
