"""The 128-pair expert tiles (k_gemm_f16.hip) at the edges of their groups of 32 pairs: tiles of one group, with the last of four
groups empty, of one pair in it, full, and of a second tile.  Weights exact in f16, activations as f16 hi and lo: 2^-22 of a factor and
the f32 order of n_in terms, 2e-5 of a row's largest output; 1e-4 through the hardware exponential of silu."""
import numpy as np
import pytest

from util import nvfp4_weights, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_in,n_out", [(256, 128), (512, 260), (1024, 64)])
@pytest.mark.parametrize("counts", [(65, 96, 97, 128), (64, 33, 129, 160), (1, 32, 63, 127), (95, 98, 192, 224)])
def test_groups_of_a_tile(counts, n_in, n_out):
    import inferred_hip as ih
    from oracle import binding as ob
    r = rng(n_in + sum(counts))
    n_expert, n_tok = len(counts), sum(counts)
    ids = r.permutation(np.repeat(np.arange(n_expert), counts)).astype(np.uint32)
    scale = [r.random(n_expert).astype(np.float32) * 0.01 + 0.002 for _ in range(2)]
    gate, up = nvfp4_weights(r, n_expert * n_out, n_in), nvfp4_weights(r, n_expert * n_out, n_in)
    x = (r.standard_normal((n_tok, n_in)) * 10.0 ** r.uniform(-2.0, 1.0, (n_tok, 1))).astype(np.float32).reshape(-1)
    be, orc = ih.Hip(exact=False), ob.Oracle(threads=8)
    try:
        be.begin_pass(n_tok)
        route = ih.Hip.host_route(ids, np.ones(n_tok, np.float32), 1)
        for what in ("glu", "single"):
            got, want, tmp, tmp2 = (np.full(n_tok * n_out, np.nan, np.float32) for _ in range(4))
            a = [ih.experts(w, ih.NVFP4, n_in, n_out, n_expert, s) for w, s in zip((gate, up), scale)]
            b = [ob.experts(w, ih.NVFP4, n_in, n_out, n_expert, s) for w, s in zip((gate, up), scale)]
            if what == "glu":
                be.moe_glu(*a, route, x, got, tmp)
                orc.moe_glu(*b, ids, 1, x, want, tmp2)
            else:
                be.matmul_experts(a[0], route, x, got)
                orc.matmul_experts(b[0], ids, 1, x, want)
            be.host_needs(got); be.raise_if_error()
            g, w = got.reshape(n_tok, n_out), want.reshape(n_tok, n_out)
            err = np.abs(g - w).max(axis=1) / np.abs(w).max(axis=1)
            assert err.max() <= (1e-4 if what == "glu" else 2e-5), (what, err.argmax(), err.max())
        be.end_pass()
    finally:
        be.take_error()
        be.close()
