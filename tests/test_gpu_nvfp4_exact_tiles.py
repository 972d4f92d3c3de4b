"""Exact mode's NVFP4 expert products over a batch, whose dots and scale products the f16 matrix instructions form: the CPU oracle's
bits at the edges of rows, slabs and tiles and over every scale code and the activation steps that f16 holds, subnormal ones included."""
import numpy as np
import pytest

from util import nvfp4_weights, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_tok,n_expert,n_used,n_in,n_out", [
    (32, 1, 1, 128, 64),       # one slab, two whole tiles
    (33, 3, 1, 256, 1),        # tiles of a few pairs, one row
    (40, 5, 2, 384, 36),
    (65, 16, 4, 640, 130),
])
@pytest.mark.parametrize("glu", [False, True])
def test_bits(n_tok, n_expert, n_used, n_in, n_out, glu):
    import inferred_hip as ih
    from oracle import binding as ob
    hip, orc = ih.Hip(exact=True), ob.Oracle(threads=8)
    r = rng(n_tok + n_in)

    def weights():
        w = nvfp4_weights(r, n_expert * n_out, n_in).reshape(-1, 36)
        w[:, :4] = r.integers(0, 256, (len(w), 4))          # every code, 0x7f (which counts as zero) and the sign bit included
        w[: len(w) // 2, :4] &= 0x3f
        return w.reshape(-1).copy()

    a, b = weights(), weights()
    scale = [r.random(n_expert).astype(np.float32) + 0.5 for _ in range(2)]
    x = r.standard_normal((n_tok, n_in // 32, 32)).astype(np.float32)
    x *= (2.0 ** r.integers(-26, 18, (n_tok, n_in // 32, 1))).astype(np.float32)      # steps of 2^-33 to 2^13
    x[0, 0] = 0
    x[1, :, 3] = 127 * 60000.0
    x = x.reshape(-1).copy()
    ids = np.stack([r.permutation(n_expert)[:n_used] for _ in range(n_tok)]).astype(np.uint32).reshape(-1)
    route = ih.Hip.host_route(ids, np.ones(len(ids), np.float32), n_used)
    got, want, other = (np.zeros(n_tok * n_used * n_out, np.float32) for _ in range(3))
    E = lambda m, data, s: m.experts(data, m.NVFP4, n_in, n_out, n_expert, s)
    try:
        if glu:
            hip.moe_glu(E(ih, a, scale[0]), E(ih, b, scale[1]), route, x, got, other.copy()); hip.host_needs(got)
            orc.moe_glu(E(ob, a, scale[0]), E(ob, b, scale[1]), ids, n_used, x, want, other)
        else:
            hip.matmul_experts(E(ih, a, scale[0]), route, x, got); hip.host_needs(got)
            orc.matmul_experts(E(ob, a, scale[0]), ids, n_used, x, want)
        hip.raise_if_error()
        finite = np.isfinite(want)
        assert finite.mean() > 0.5 and np.array_equal(finite, np.isfinite(got))
        assert np.array_equal(got[finite].view(np.uint32), want[finite].view(np.uint32))
    finally:
        hip.take_error()
        hip.close()
