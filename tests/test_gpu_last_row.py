"""The output matrix on a batch pass's last row (gather, norm, quantization and product as one launch): against the CPU oracle, in the
first pass, whose buffers still have to grow, and in later ones, which must give the same bits; with a factor behind it; and left as it
is where an op behind it reads the gathered row or multiplies the normed one again."""
import numpy as np
import pytest

from util import bound, q8_0_weights, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("then", ["nothing", "scale", "reads the row", "second product"])
@pytest.mark.parametrize("nd,n_vocab,n", [(256, 70, 2), (2048, 515, 23), (4096, 64, 40), (1024, 33, 300)])
def test_last_row(nd, n_vocab, n, then):
    import inferred_hip as ih
    from oracle import binding as ob
    orc, hip = ob.Oracle(threads=4), ih.Hip(exact=False)
    r = rng(nd + n)
    data, data2 = (q8_0_weights(orc, r, n_vocab, nd, std=nd ** -0.5) for _ in range(2))
    W, W2 = ([m.weights(d, ih.Q8_0, nd, n_vocab) for m in (ih, ob)] for d in (data, data2))
    norm = (0.5 + r.random(nd)).astype(np.float32)
    B = [dict(x=np.zeros(n * nd, np.float32), last=np.zeros(nd, np.float32), normed=np.zeros(nd, np.float32), sum=np.zeros(nd, np.float32),
              logits=np.zeros(n_vocab, np.float32), more=np.zeros(n_vocab, np.float32)) for _ in range(2)]

    def tail(ops, i, b):
        ops.gather_chunks(b["x"], nd, nd, (n - 1) * nd, b["last"])
        ops.rms_norm(b["last"], norm, 1e-6, b["normed"])
        ops.matmul(W[i], b["normed"], b["logits"])
        if then == "scale":
            ops.scale(b["logits"], 0.375)
        if then == "reads the row":
            ops.add_assign(b["sum"], b["last"])
        if then == "second product":
            ops.matmul(W2[i], b["normed"], b["more"])

    outs = []
    try:
        for p in range(3):
            x = rng(9).standard_normal(n * nd).astype(np.float32)
            for b in B:
                b["x"][:], b["sum"][:] = x, 0
            hip.begin_pass(n); hip.host_wrote(B[0]["x"]); hip.host_wrote(B[0]["sum"])
            tail(hip, 0, B[0])
            hip.end_pass()
            got = [B[0][k] for k in ("logits", "normed") + (("sum",) if then == "reads the row" else ("more",) if then == "second product" else ())]
            for g in got:
                hip.host_needs(g)
            hip.raise_if_error()
            outs.append([g.copy() for g in got])
        tail(orc, 1, B[1])
        want = [B[1][k] for k in ("logits", "normed") + (("sum",) if then == "reads the row" else ("more",) if then == "second product" else ())]
        for o in outs:
            for g, w, first in zip(o, want, outs[0]):
                assert (np.abs(g - w) <= bound(w, 1e-4)).all()        # sums in wave order: 2^-24 of nd / 32 terms
                assert np.array_equal(g.view(np.uint32), first.view(np.uint32))
    finally:
        hip.take_error()
        hip.close()
