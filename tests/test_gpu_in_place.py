"""Runs of ops that write one of their own inputs: the fused launches, whose blocks read the whole activation at their own time,
leave them to the ops.  Against the CPU oracle, bits in exact mode; fast mode's sums in wave order differ by 2^-24 of nd / 32 terms,
and by a Q8_0 step where that moves one."""
import numpy as np
import pytest

from util import bound, q8_0_weights, rng

pytestmark = pytest.mark.gpu


def norm_in_place(ops, w, b, norm):
    ops.rms_norm(b["x"], norm, 1e-6, b["x"])
    ops.matmul(w, b["x"], b["out"])


def over_the_residual(ops, w, b, norm):
    ops.rms_norm(b["x"], norm, 1e-6, b["out"])
    ops.matmul(w, b["out"], b["x"])


def over_its_input(ops, w, b, norm):
    ops.matmul(w, b["x"], b["x"])


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("run", [norm_in_place, over_the_residual, over_its_input])
@pytest.mark.parametrize("nd,n", [(256, 1), (2048, 1), (2048, 23)])
def test_own_input(nd, n, run, exact):
    import inferred_hip as ih
    from oracle import binding as ob
    orc, hip = ob.Oracle(threads=4), ih.Hip(exact=exact)
    r = rng(nd)
    data = q8_0_weights(orc, r, nd, nd, std=nd ** -0.5)
    W = [m.weights(data, ih.Q8_0, nd, nd) for m in (ih, ob)]
    norm = (0.5 + r.random(nd)).astype(np.float32)
    B = [dict(src=np.zeros(n * nd, np.float32), x=np.zeros(nd, np.float32), out=np.zeros(nd, np.float32)) for _ in range(2)]
    try:
        for p in range(5):                  # op by op, recorded and replayed (one token); the row of a batch pass
            for b in B:
                b["src"][:] = rng(9 + p).standard_normal(n * nd)
            hip.begin_pass(n); hip.host_wrote(B[0]["src"])
            for ops, i in ((hip, 0), (orc, 1)):
                ops.gather_chunks(B[i]["src"], nd, nd, (n - 1) * nd, B[i]["x"])
                run(ops, W[i], B[i], norm)
            hip.end_pass()
            for name in ("x",) if run is over_its_input else ("x", "out"):
                hip.host_needs(B[0][name])
                got, want = B[0][name], B[1][name]
                if exact:
                    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (p, name)
                else:
                    assert (np.abs(got - want) <= bound(want, 1e-4)).all(), (p, name)
            hip.raise_if_error()
    finally:
        hip.take_error()
        hip.close()
