"""The exact delta rule over a batch at the edges of its chunks of sixteen tokens and of its blocks of sixteen rows (its read-out is
added up by another wave, a token behind), against the CPU oracle bit for bit, the state carried into a second call."""
import numpy as np
import pytest

from util import assert_bits_equal, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_tok", [2, 15, 16, 17, 33, 64])
@pytest.mark.parametrize("dk,dv,nk,nv", [(32, 16, 1, 1), (64, 40, 2, 4), (128, 128, 1, 3)])
def test_chunks(n_tok, dk, dv, nk, nv):
    import inferred_hip as ih
    from oracle import binding as ob
    hip, orc = ih.Hip(exact=True), ob.Oracle(threads=4)
    r = rng(n_tok + dk)
    draw = lambda n, s=1.0: (r.standard_normal(n) * s).astype(np.float32)
    ssm_a, dt = -np.abs(draw(nv)), draw(nv)
    sa = draw(nv * dv * dk, 0.1)
    sb = sa.copy()
    try:
        for call in range(2):
            q, k, v = draw(n_tok * nk * dk, dk ** -0.5), draw(n_tok * nk * dk, dk ** -0.5), draw(n_tok * nv * dv)
            alpha, beta = draw(n_tok * nv), draw(n_tok * nv)
            a, b = np.zeros(n_tok * nv * dv, np.float32), np.zeros(n_tok * nv * dv, np.float32)
            hip.begin_pass(n_tok)
            hip.delta_rule(q, k, v, alpha, beta, ssm_a, dt, dk, dv, nk, nv, sa, a)
            hip.end_pass(); hip.host_needs(a); hip.read_state(sa); hip.raise_if_error()
            orc.delta_rule(q, k, v, alpha, beta, ssm_a, dt, dk, dv, nk, nv, sb, b)
            assert_bits_equal(a, b, f"out, call {call}")
            assert_bits_equal(sa, sb, f"state, call {call}")
    finally:
        hip.take_error()
        hip.close()
