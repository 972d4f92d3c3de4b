"""The routed FFN where its ops take different kernels: which of them sorts the pairs by experts for the next."""
import numpy as np
import pytest

from util import q8_0_weights, rng

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def orc():
    from oracle import binding as ob
    return ob.Oracle(threads=8)


@pytest.fixture(scope="module")
def pair():
    import inferred_hip as ih
    two = [ih.Hip(exact=False, fuse=True), ih.Hip(exact=False, fuse=False)]
    yield two
    errs = [be.take_error() for be in two]
    for be in two:
        be.close()
    assert errs == [None, None], errs


def z(k):
    return np.zeros(k, np.float32)


@pytest.mark.parametrize("nd,ff", [(1056, 512), (512, 1056)])
def test_products_of_which_one_kernel_groups_and_the_other_does_not(pair, orc, nd, ff):
    """Q8_0 experts with rows of 33 blocks run one GEMV a pair, those with rows of 16 the tiles of the same route: against the
    CPU oracle (only the order of the sums differs, and silu's exponential: 1e-4 of a row's largest value)."""
    import inferred_hip as ih
    from oracle import binding as ob
    n, ne, nu, be = 40, 8, 2, pair[0]
    r = rng(12)
    gate, up, down = (q8_0_weights(orc, r, ne * o, i, std=0.05) for o, i in ((ff, nd), (ff, nd), (nd, ff)))
    x, probs = r.standard_normal(n * nd).astype(np.float32), r.standard_normal(n * ne).astype(np.float32)
    g, u, o, pa = z(n * nu * ff), z(n * nu * ff), z(n * nu * nd), probs.copy()
    go, uo, oo, pb = z(n * nu * ff), z(n * nu * ff), z(n * nu * nd), probs.copy()
    be.drop_mirrors()
    be.begin_pass(n)
    be.host_wrote(x); be.host_wrote(pa)
    be.softmax(pa, ne)
    route = be.route(pa, ne, nu)
    be.moe_glu(ih.experts(gate, ih.Q8_0, nd, ff, ne, None), ih.experts(up, ih.Q8_0, nd, ff, ne, None), route, x, g, u)
    be.matmul_experts(ih.experts(down, ih.Q8_0, ff, nd, ne, None), route, g, o)
    be.end_pass()
    be.host_needs(g); be.host_needs(o)
    be.raise_if_error()
    orc.softmax(pb, ne)
    ids, _ = orc.route(pb, ne, nu)
    orc.moe_glu(ob.experts(gate, ob.Q8_0, nd, ff, ne, None), ob.experts(up, ob.Q8_0, nd, ff, ne, None), ids, nu, x, go, uo)
    orc.matmul_experts(ob.experts(down, ob.Q8_0, ff, nd, ne, None), ids, nu, g, oo)   # of the backend's own gate / up product
    for a, b in ((g, go), (o, oo)):
        a, b = a.reshape(n * nu, -1), b.reshape(n * nu, -1)
        assert (np.abs(a - b) <= 1e-4 * np.abs(b).max(1, keepdims=True)).all()
