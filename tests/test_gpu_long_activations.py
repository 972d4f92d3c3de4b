"""Single-token passes over activations as long as a wave of the fused products takes a row at once (16,384 values) and over longer ones, which
are issued op by op: both modes against the CPU oracle, op by op, recorded and replayed."""
import numpy as np
import pytest

from util import close, q8_0_weights, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("n_in,fused", [(16352, True), (16384, True), (16416, False), (18368, False), (20512, False), (22528, False)])
def test_product_added_to_a_residual(exact, n_in, fused):
    import inferred_hip as ih
    from oracle import binding as ob
    orc = ob.Oracle(threads=8)
    hip = ih.Hip(exact=exact)
    n_out = 70
    r = rng(n_in)
    data = q8_0_weights(orc, r, n_out, n_in, std=n_in ** -0.5)
    W = [m.weights(data, ih.Q8_0, n_in, n_out) for m in (ih, ob)]
    B = [dict(x=np.zeros(n_in, np.float32), y=np.zeros(n_out, np.float32), res=np.zeros(n_out, np.float32)) for _ in range(2)]

    def block(ops, w, b):
        ops.matmul(w, b["x"], b["y"])
        ops.add_assign(b["res"], b["y"])

    try:
        for p in range(5):
            fresh = rng(n_in + p)
            x0, r0 = fresh.standard_normal(n_in).astype(np.float32), fresh.standard_normal(n_out).astype(np.float32)
            for b in B:
                b["x"][:], b["res"][:] = x0, r0
            hip.begin_pass(1); hip.host_wrote(B[0]["x"]); hip.host_wrote(B[0]["res"])
            block(hip, W[0], B[0])
            hip.end_pass(); hip.host_needs(B[0]["res"]); hip.raise_if_error()
            block(orc, W[1], B[1])
            got, want = B[0]["res"], B[1]["res"]
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)) if exact else close(got, want), p
        g = hip.graph_stats()
        assert g["captures"] == 1 and g["replays"] == 3 and g["graph_kernels"] == (1 if fused else 3), g
    finally:
        hip.take_error()
        hip.close()
