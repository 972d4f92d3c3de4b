"""The output matrix on a batch pass's last row (gather, norm, quantization and product as one launch): against the CPU oracle, in the
first pass, whose buffers still have to grow, and in later ones, which must give the same bits; with a factor behind it; where the
gathered row is read by the next op, by one behind it or by the host; where the norm replaces it; and left as it is where an op
behind multiplies the normed row again.  The same of a single-token pass, recorded and replayed."""
import numpy as np
import pytest

from util import bound, nvfp4_weights, q8_0_weights, rng

pytestmark = pytest.mark.gpu
SHAPES = [(256, 70, 2), (2048, 515, 23), (4096, 64, 40), (1024, 33, 300)]
NAMES = ("logits", "normed", "last", "sum", "more")


class Tail:
    def __init__(self, fmt, nd, n_vocab, n, then):
        import inferred_hip as ih
        from oracle import binding as ob
        self.orc = ob.Oracle(threads=4)
        self.nd, self.n, self.then = nd, n, then
        r = rng(nd + n)
        draw = (lambda: nvfp4_weights(r, n_vocab, nd)) if fmt == "nvfp4" else (lambda: q8_0_weights(self.orc, r, n_vocab, nd, std=nd ** -0.5))
        self.data = [draw() for _ in range(2)]
        ty = ih.NVFP4 if fmt == "nvfp4" else ih.Q8_0
        self.W, self.W2 = ([m.weights(d, ty, nd, n_vocab) for m in (ih, ob)] for d in self.data)
        self.norm = (0.5 + r.random(nd)).astype(np.float32)
        self.B = [dict(x=np.zeros(n * nd, np.float32), last=np.zeros(nd, np.float32), normed=np.zeros(nd, np.float32), sum=np.zeros(nd, np.float32),
                       logits=np.zeros(n_vocab, np.float32), more=np.zeros(n_vocab, np.float32)) for _ in range(2)]

    def ops(self, ops, i):
        b, then = self.B[i], self.then
        normed = b["last"] if then == "norm in place" else b["normed"]
        ops.gather_chunks(b["x"], self.nd, self.nd, (self.n - 1) * self.nd, b["last"])
        ops.rms_norm(b["last"], self.norm, 1e-6, normed)
        ops.matmul(self.W[i], normed, b["logits"])
        if then == "scale":
            ops.scale(b["logits"], 0.375)
        if then == "reads the row later":
            ops.scale(b["logits"], 0.375)
            ops.scale(b["sum"], 2.0)
        if then in ("reads the row", "reads the row later"):
            ops.add_assign(b["sum"], b["last"])
        if then == "second product":
            ops.matmul(self.W2[i], normed, b["more"])

    def start(self, hip, p):
        x = rng(9 + p).standard_normal(self.n * self.nd).astype(np.float32)
        for b in self.B:
            b["x"][:], b["sum"][:] = x, 1.5
        hip.begin_pass(self.n)
        hip.host_wrote(self.B[0]["x"]); hip.host_wrote(self.B[0]["sum"])

    def read(self, hip):
        names = [n for n in NAMES if n in ("logits", "last") or (n == "normed" and self.then != "norm in place")
                 or (n == "sum" and "reads" in self.then) or (n == "more" and self.then == "second product")]
        for name in names:
            hip.host_needs(self.B[0][name])
        hip.raise_if_error()
        return {name: self.B[0][name].copy() for name in names}

    def check(self, got):
        self.ops(self.orc, 1)
        for name, g in got.items():
            want = self.B[1][name]
            if name in ("last", "sum") and self.then != "norm in place":
                assert np.array_equal(g.view(np.uint32), want.view(np.uint32)), name    # copies and one addition
            else:
                assert (np.abs(g - want) <= bound(want, 1e-4)).all(), name    # sums in wave order: 2^-24 of nd / 32 terms


@pytest.mark.parametrize("fmt", ["q8", "nvfp4"])
@pytest.mark.parametrize("then", ["nothing", "scale", "reads the row", "reads the row later", "norm in place", "second product"])
@pytest.mark.parametrize("nd,n_vocab,n", SHAPES)
def test_last_row(nd, n_vocab, n, then, fmt):
    import inferred_hip as ih
    hip = ih.Hip(exact=False)
    t = Tail(fmt, nd, n_vocab, n, then)
    try:
        outs = []
        for p in range(3):
            t.start(hip, 0)
            if p == 2:
                hip.profile_begin()
            t.ops(hip, 0)
            hip.end_pass()
            if p == 2:
                heads = [r["launches"] for r in hip.profile_end() if r["name"].startswith("lm_head")]
                assert heads == ([] if then == "second product" else [1]), heads      # (one launch, or op by op)
            outs.append(t.read(hip))
        for o in outs:
            t.start(hip, 0)
            t.check(o)
            for name, g in o.items():
                assert np.array_equal(g.view(np.uint32), outs[0][name].view(np.uint32)), name
    finally:
        hip.take_error()
        hip.close()


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("then", ["nothing", "reads the row", "norm in place"])
@pytest.mark.parametrize("nd,n_vocab", [(256, 70), (2048, 515), (5120, 64)])
def test_single_token(nd, n_vocab, then, exact):
    import inferred_hip as ih
    hip = ih.Hip(exact=exact, chain=False)
    t = Tail("q8", nd, n_vocab, 1, then)
    try:
        for p in range(6):
            t.start(hip, p)
            t.ops(hip, 0)
            hip.end_pass()
            t.check(t.read(hip))
        g = hip.graph_stats()
        assert g["captures"] == 1 and g["replays"] >= 2 and g["graph_kernels"] == (2 if then == "reads the row" else 1), g
    finally:
        hip.take_error()
        hip.close()
