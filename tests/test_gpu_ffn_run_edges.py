"""The routed FFN of a short batch as two launches (fuser.cpp, small_ffn), with ops behind it that use what the run leaves
out: the route's grouping by experts, the quantized and split forms of its rows, the buffers its kernels do not write.  The
same ops on a backend with fusion off are the reference; the two differ in the order of f32 sums and in the Q8_0 steps that
this moves (1/127 of a block's largest value each, a few of a row), so 1e-2 of a result's 2-norm bounds them, where a form or
a grouping left over from another pass gives about 1.
"""
import numpy as np
import pytest

from util import nvfp4_weights, q8_0_weights, rng

pytestmark = pytest.mark.gpu
ND, FF, NE, NU, N = 512, 256, 32, 8, 8


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


class Ffn:
    def __init__(self, orc, nd=ND, ff=FF, ne=NE, code=None, seed=5):
        import inferred_hip as ih
        r = rng(seed)
        code = ih.NVFP4 if code is None else code
        self.ih, self.nd, self.ff, self.ne, self.keep = ih, nd, ff, ne, []
        rows = lambda n_out, n_in: self.hold(nvfp4_weights(r, n_out, n_in) if code == ih.NVFP4 else q8_0_weights(orc, r, n_out, n_in, std=0.05))  # noqa: E731
        q8 = lambda n_out, n_in: ih.weights(self.hold(q8_0_weights(orc, r, n_out, n_in, std=0.05)), ih.Q8_0, n_in, n_out)  # noqa: E731
        sc = lambda: self.hold((0.5 + r.random(ne)).astype(np.float32) / 16) if code == ih.NVFP4 else None  # noqa: E731
        self.gate, self.up = (ih.experts(rows(ne * ff, nd), code, nd, ff, ne, sc()) for _ in range(2))
        self.down = ih.experts(rows(ne * nd, ff), code, ff, nd, ne, sc())
        self.router, self.logit, self.sg, self.su, self.sd = q8(ne, nd), q8(1, nd), q8(ff, nd), q8(ff, nd), q8(nd, ff)
        self.w64, self.w64_ff = q8(64, nd), q8(64, ff)

    def hold(self, a):
        self.keep.append(a)
        return a

    def run(self, be, b, nu):
        """the block from the router product to the combine; returns the route"""
        be.matmul_pair(self.router, self.logit, b["x"], b["router"], b["logit"])
        be.softmax(b["router"], self.ne)
        route = be.route(b["router"], self.ne, nu)
        be.moe_glu(self.gate, self.up, route, b["x"], b["g"], b["u"])
        be.matmul_experts(self.down, route, b["g"], b["o"])
        be.matmul(self.sg, b["x"], b["e_gate"])
        be.matmul(self.su, b["x"], b["e_up"])
        be.silu_mul(b["e_gate"], b["e_up"])
        be.matmul(self.sd, b["e_gate"], b["e_out"])
        be.moe_finish(b["y"], 0, self.nd, b["o"], route, b["e_out"], b["logit"], 0)
        return route


def buffers(r, n, nu, ffn):
    nd, ff, ne = ffn.nd, ffn.ff, ffn.ne
    return dict(x=(r.standard_normal(n * nd)).astype(np.float32), router=z(n * ne), logit=z(n), g=z(n * nu * ff), u=z(n * nu * ff), o=z(n * nu * nd),
                e_gate=z(n * ff), e_up=z(n * ff), e_out=z(n * nd), y=z(n * nd), router2=z(n * ne), logit2=z(n), g2=z(n * nu * ff), o2=z(n * nu * nd), out=z(n * 64),
                acc=z(n * nd))


def compare(pair, n, b0, script, outs, taken):
    got, launches = [], []
    for be in pair:
        be.drop_mirrors()
        b = {k: v.copy() for k, v in b0.items()}
        for rep in range(2):   # the first pass sizes the mirrors, which ends a held run, and leaves other values behind
            b["x"][:] = b0["x"] if rep else -0.5 * b0["x"][::-1]
            be.begin_pass(n)
            be.host_wrote(b["x"])
            if rep:
                be.profile_begin()
            script(be, b)
            be.end_pass()
            if rep:
                launches.append(sum(r["launches"] for r in be.profile_end()))
        for o in outs:
            be.host_needs(b[o])
        be.raise_if_error()
        got.append(b)
    for o in outs:
        want = got[1][o].astype(np.float64)
        assert np.isfinite(got[0][o]).all(), o
        err = np.linalg.norm(got[0][o] - want) / max(np.linalg.norm(want), 1e-30)
        print(o, err, launches, flush=True)
        assert err <= 1e-2, (o, err)
    # a run that is taken has ten ops in two launches; one that is not has softmax and route in one
    assert (launches[0] <= launches[1] - 8) == taken, launches


@pytest.mark.parametrize("n", [3, 4, 8, 32])
@pytest.mark.parametrize("same_route", [True, False])
def test_further_expert_products_behind_the_run(pair, orc, n, same_route):
    """They need the rows' split form, and on the same route the pairs grouped by experts: the run makes neither."""
    ffn = Ffn(orc)

    def script(be, b):
        route = ffn.run(be, b, NU)
        if not same_route:
            be.matmul_pair(ffn.router, ffn.logit, b["x"], b["router2"], b["logit2"])
            be.scale(b["router2"], -1.0)
            be.softmax(b["router2"], NE)
            route = be.route(b["router2"], NE, NU)
        be.moe_glu(ffn.gate, ffn.up, route, b["x"], b["g2"], b["u"])
        be.matmul_experts(ffn.down, route, b["g2"], b["o2"])
    compare(pair, n, buffers(rng(11), n, NU, ffn), script, ["y", "g2", "o2"], True)


BEHIND = {   # an op right behind the run, and the outputs to compare
    "product_on_the_rows": lambda f, be, b: be.matmul(f.w64, b["x"], b["out"]),
    "product_on_the_gated_rows": lambda f, be, b: be.matmul(f.w64_ff, b["e_gate"], b["out"]),
    "sum_of_the_picks": lambda f, be, b: be.add_scaled_rows(b["acc"], b["o"], b["pick_w"]),
    "probabilities": lambda f, be, b: be.gather_chunks(b["router"], NE, NE, 0, b["router2"]),
    "probabilities_changed": lambda f, be, b: be.scale(b["router"], 2.0),
    "up_product": lambda f, be, b: be.scatter_chunks(b["e_up"], FF, FF, 0, b["acc"]),
    "new_probabilities": lambda f, be, b: be.matmul(f.router, b["y"], b["router"]),
}


@pytest.mark.parametrize("what", sorted(BEHIND))
@pytest.mark.parametrize("n", [3, 8])
def test_an_op_behind_that_uses_what_the_run_leaves_out(pair, orc, n, what):
    ffn = Ffn(orc)
    b = buffers(rng(15), n, NU, ffn)
    if what == "product_on_the_rows":   # an F32 router: the rows are quantized for the experts, inside the run
        for name, rows in (("router", NE), ("logit", 1)):
            w = ffn.hold((rng(17).standard_normal(rows * ND) * 0.1).astype(np.float32))
            setattr(ffn, name, ffn.ih.weights(w.view(np.uint8), ffn.ih.F32, ND, rows))
    if what == "sum_of_the_picks":
        b.update(pick_w=rng(16).standard_normal(n * NU).astype(np.float32), acc=z(ND))

    def script(be, b):
        if "pick_w" in b:
            be.host_wrote(b["pick_w"])
        ffn.run(be, b, NU)
        BEHIND[what](ffn, be, b)
    compare(pair, n, b, script, ["y", "out", "acc", "router2"] + (["router"] if "probabilities_" in what or "new" in what else []), False)


@pytest.mark.parametrize("n", [8, 32])
def test_rows_in_a_buffer_that_has_only_been_quantized_before(pair, orc, n):
    """A run that reads no split form does not wait for room for one."""
    ffn, be = Ffn(orc), pair[0]
    be.drop_mirrors()
    b = buffers(rng(14), n, NU, ffn)
    rows = [b["x"].copy() for _ in range(3)]
    for i, x in enumerate(rows):
        b["x"] = x
        for whole in (False, True):
            be.begin_pass(n)
            be.host_wrote(x)
            if whole:
                be.profile_begin()
                ffn.run(be, b, NU)
            else:
                be.matmul(ffn.w64, x, b["out"])
            be.end_pass()
        launches = sum(r["launches"] for r in be.profile_end())
        be.raise_if_error()
    assert launches <= 5, launches   # the rows' form, two router products, the run


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
