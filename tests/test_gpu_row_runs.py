"""Runs of row-wise ops of a batch pass that fast mode issues as one kernel each (k_rows.hip, fuser.cpp), against the same ops
issued one by one by a backend with fusion off: the residual row (moe_finish, add, rms norm, copy and the Q8_0 form), the gate
and quantization in front of a product, softmax with the routing decision, attention's rows before the scores, and the NVFP4
shared expert's gate / up pair.  The kernels form every value as the separate ones do but for the order of the long sums, so
the two agree to rounding (products of quantized rows: to a quant or two of the row).  Sizes at the edges of what a wave, a
block or a tile holds; the number of launches says that the run was taken.
"""
import numpy as np
import pytest

from util import close, nvfp4_weights, q8_0_weights, rng, worst

pytestmark = pytest.mark.gpu
EPS = 1e-6


@pytest.fixture(scope="module")
def pair():
    import inferred_hip as ih
    two = [ih.Hip(exact=False, fuse=True), ih.Hip(exact=False, fuse=False)]
    yield two
    errs = [be.take_error() for be in two]
    for be in two:
        be.close()
    assert errs == [None, None], errs


@pytest.fixture(scope="module")
def orc():
    from oracle import binding as ob
    return ob.Oracle(threads=8)


def run(pair, n, bufs, script, outs, tol=1e-5, at_most=None, other_first=False):
    """other_first: the first pass has other values, so that what it leaves behind cannot pass for the second's."""
    got = []
    for be in pair:
        be.drop_mirrors()
        b = {k: v.copy() for k, v in bufs.items()}
        for rep in range(2):   # twice: the first pass sizes the mirrors, which ends runs early
            for k, v in bufs.items():
                b[k][...] = v if rep or not other_first else -0.5 * v[::-1]
            be.begin_pass(n)
            for v in b.values():
                if v.dtype == np.float32:
                    be.host_wrote(v)
            if rep:
                be.profile_begin()
            script(be, b)
            be.end_pass()
            if rep:
                launches = sum(r["launches"] for r in be.profile_end())
        for o in outs:
            be.host_needs(b[o])
        be.raise_if_error()
        got.append((b, launches))
    for o in outs:
        assert close(got[0][0][o], got[1][0][o], tol), (o, worst(got[0][0][o], got[1][0][o]))
    if at_most is not None:
        assert got[0][1] <= at_most < got[1][1], (got[0][1], got[1][1])
    return got


def q8_0_weights_of(r, n_out, n_in):
    from oracle import binding as ob
    return q8_0_weights(ob.Oracle(threads=2), r, n_out, n_in, std=0.05)


def f32(r, k, s=1.0):
    return (r.standard_normal(k) * s).astype(np.float32)


@pytest.mark.parametrize("n,nd", [(2, 1024), (3, 1056), (5, 2048), (33, 4096), (2, 4128), (3, 8192)])
def test_the_residual_row(pair, orc, n, nd):
    import inferred_hip as ih
    r = rng(1)
    w = q8_0_weights(orc, r, 64, nd, std=0.05)
    norm = (0.5 + r.random(nd)).astype(np.float32)
    b = dict(x=f32(r, n * nd), y=f32(r, n * nd), normed=np.zeros(n * nd, np.float32), copy=np.zeros(n * nd, np.float32),
             out=np.zeros(n * 64, np.float32), out2=np.zeros(n * 64, np.float32))

    def script(be, b):
        be.add_assign(b["x"], b["y"])
        be.rms_norm(b["x"], norm, EPS, b["normed"])
        be.gather_chunks(b["normed"], n * nd, n * nd, 0, b["copy"])
        be.matmul(ih.weights(w, ih.Q8_0, nd, 64), b["copy"], b["out"])
        be.matmul(ih.weights(w, ih.Q8_0, nd, 64), b["normed"], b["out2"])   # the normed rows are still there for others
    run(pair, n, b, script, ["x", "normed", "copy"], at_most=5)
    run(pair, n, b, script, ["out", "out2"], tol=3e-2)


@pytest.mark.parametrize("what", ["normed_first", "normed_first_nvfp4", "into_the_copy", "part_of_the_copy", "scatter_into_the_copy"])
@pytest.mark.parametrize("n,nd", [(3, 1024), (40, 2048)])
def test_the_residual_row_in_front_of_other_readers_and_writers(pair, orc, n, nd, what):
    """The op behind the run had its pointers taken before the run was issued: one that reads the normed rows' Q8_0 form, one
    that writes the copy, one that reads a part of the copy (whose form has less room than the whole one needs).  Every
    product is compared with the one of the backend that issues the ops one by one."""
    import inferred_hip as ih
    r = rng(7)
    w, sq = q8_0_weights(orc, r, 64, nd, std=0.05), q8_0_weights(orc, r, nd, nd, std=0.05)
    w4 = nvfp4_weights(r, 64, nd)
    norm = (0.5 + r.random(nd)).astype(np.float32)
    z = lambda k: np.zeros(k, np.float32)  # noqa: E731
    b = dict(x=f32(r, n * nd), y=f32(r, n * nd), z=f32(r, n * nd), normed=z(n * nd), copy=z(n * nd), out=z(n * 64), out2=z(n * 64))
    w64 = ih.weights(w, ih.Q8_0, nd, 64)

    def script(be, b):
        be.add_assign(b["x"], b["y"])
        be.rms_norm(b["x"], norm, EPS, b["normed"])
        be.gather_chunks(b["normed"], n * nd, n * nd, 0, b["copy"])
        if what == "normed_first":
            be.matmul(w64, b["normed"], b["out2"])
        elif what == "normed_first_nvfp4":
            be.matmul(ih.weights(w4, ih.NVFP4, nd, 64), b["normed"], b["out2"])
        elif what == "into_the_copy":
            be.matmul(ih.weights(sq, ih.Q8_0, nd, nd), b["z"], b["copy"])
        elif what == "part_of_the_copy":
            be.matmul(w64, b["copy"][:nd], b["out2"][:64])
            return   # (the form of the whole copy is never asked for)
        else:
            be.scatter_chunks(b["z"], n * nd, n * nd, 0, b["copy"])
        be.matmul(w64, b["copy"], b["out"])
    run(pair, n, b, script, ["x", "normed", "copy", "out", "out2"], tol=3e-2, other_first=True)


@pytest.mark.parametrize("n,nd,nu", [(2, 1024, 4), (3, 2048, 10), (5, 1056, 3), (40, 2048, 8)])
def test_the_routed_sum_in_front_of_the_residual(pair, n, nd, nu):
    r = rng(2)
    ne = 32
    norm = (0.5 + r.random(nd)).astype(np.float32)
    b = dict(probs=f32(r, n * ne), rows=f32(r, n * nu * nd), shared=f32(r, n * nd), logit=f32(r, n), x=f32(r, n * nd),
             y=np.zeros(n * nd, np.float32), normed=np.zeros(n * nd, np.float32))

    def script(be, b):
        be.softmax(b["probs"], ne)
        route = be.route(b["probs"], ne, nu)
        be.moe_finish(b["y"], 0, nd, b["rows"], route, b["shared"], b["logit"], 0)
        be.add_assign(b["x"], b["y"])
        be.rms_norm(b["x"], norm, EPS, b["normed"])
    run(pair, n, b, script, ["probs", "y", "x", "normed"], at_most=2)


@pytest.mark.parametrize("n,width", [(2, 32), (3, 256), (5, 288), (2, 1024), (7, 1056), (2, 2080), (3, 4096), (2, 8192)])
def test_a_gate_and_the_quantized_product_behind_it(pair, orc, n, width):
    import inferred_hip as ih
    r = rng(3)
    w = q8_0_weights(orc, r, 32, width, std=0.05)
    b = dict(x=f32(r, n * width), g=f32(r, n * width), out=np.zeros(n * 32, np.float32))

    def script(be, b):
        be.sigmoid_mul(b["x"], b["g"])
        be.matmul(ih.weights(w, ih.Q8_0, width, 32), b["x"], b["out"])
    run(pair, n, b, script, ["x"], at_most=2)
    run(pair, n, b, script, ["out"], tol=3e-2)


@pytest.mark.parametrize("n,ne,nu", [(2, 16, 1), (5, 64, 16), (3, 100, 4), (67, 512, 10), (2, 1000, 10), (3, 1024, 16)])
def test_softmax_and_route(pair, n, ne, nu):
    r = rng(4)
    b = dict(probs=f32(r, n * ne, 2.0), rows=f32(r, n * nu * 32), shared=np.zeros(n * 32, np.float32), logit=np.zeros(n, np.float32),
             y=np.zeros(n * 32, np.float32))
    b["probs"].reshape(n, ne)[0, : ne // 2] = 1.5     # ties go to the lower id

    def script(be, b):
        be.softmax(b["probs"], ne)
        route = be.route(b["probs"], ne, nu)
        be.moe_finish(b["y"], 0, 32, b["rows"], route, b["shared"], b["logit"], 0)
    run(pair, n, b, script, ["probs", "y"], at_most=2)


@pytest.mark.parametrize("n,hd,n_rot,nh,nkv", [(2, 64, 64, 4, 2), (3, 128, 32, 8, 2), (65, 256, 64, 16, 2), (7, 256, 256, 4, 4)])
def test_attentions_rows(pair, orc, n, hd, n_rot, nh, nkv):
    import inferred_hip as ih
    r = rng(5)
    qw, kw = (0.5 + r.random(hd)).astype(np.float32), (0.5 + r.random(hd)).astype(np.float32)
    nd, pos, ctx = 64, 11, 128
    wk, wv = (q8_0_weights(orc, r, nkv * hd, nd, std=0.2) for _ in range(2))
    z = lambda k: np.zeros(k, np.float32)  # noqa: E731
    b = dict(qg=f32(r, n * nh * 2 * hd), h=f32(r, n * nd), q=z(n * nh * hd), g=z(n * nh * hd), k=z(n * nkv * hd), v=z(n * nkv * hd))
    slabs = [[np.zeros(ctx * nkv * hd, np.uint16) for _ in range(2)] for _ in pair]

    def script(be, b):
        sk, sv = slabs[0 if be is pair[0] else 1]
        be.matmul(ih.weights(wk, ih.Q8_0, nd, nkv * hd), b["h"], b["k"])     # (the rows are quantized before the run, as a layer's are)
        be.gather_chunks(b["qg"], hd, 2 * hd, 0, b["q"])
        be.gather_chunks(b["qg"], hd, 2 * hd, hd, b["g"])
        be.matmul(ih.weights(wk, ih.Q8_0, nd, nkv * hd), b["h"], b["k"])
        be.matmul(ih.weights(wv, ih.Q8_0, nd, nkv * hd), b["h"], b["v"])
        be.rms_norm_heads(b["q"], qw, hd, EPS)
        be.rms_norm_heads(b["k"], kw, hd, EPS)
        be.rope_neox(b["q"], pos, hd, n_rot, nh, 1e6)
        be.rope_neox(b["k"], pos, hd, n_rot, nkv, 1e6)
        be.kv_write(sk, pos * nkv * hd, b["k"])
        be.kv_write(sv, pos * nkv * hd, b["v"])
    run(pair, n, b, script, ["q", "g", "k", "v"], at_most=5)
    for be, (sk, sv) in zip(pair, slabs):
        be.read_kv(sk)
        be.read_kv(sv)
    for a, c in zip(*slabs):
        fa, fc = a.view(np.float16).astype(np.float32), c.view(np.float16).astype(np.float32)
        assert close(fa, fc, 2e-3), worst(fa, fc)
        assert np.array_equal(np.flatnonzero(fa), np.flatnonzero(fc))


@pytest.mark.parametrize("n,nd,ff", [(128, 512, 64), (131, 768, 68), (1024, 256, 128), (1030, 512, 96)])
def test_the_nvfp4_shared_expert(pair, n, nd, ff):
    """16-wide tiles up to 1,024 tokens (row lengths with and without a split of k over the waves), 128-wide above."""
    import inferred_hip as ih
    r = rng(6)
    wg, wu, wd = nvfp4_weights(r, ff, nd), nvfp4_weights(r, ff, nd), nvfp4_weights(r, nd, 256)
    z = lambda k: np.zeros(k, np.float32)  # noqa: E731
    b = dict(x=f32(r, n * nd, 0.2), gate=z(n * ff), up=z(n * ff), h=f32(r, n * 256, 0.2), out=z(n * nd))

    def script(be, b):
        be.matmul(ih.weights(wg, ih.NVFP4, nd, ff), b["x"], b["gate"])
        be.matmul(ih.weights(wu, ih.NVFP4, nd, ff), b["x"], b["up"])
        be.scale(b["up"], 0.25)
        be.scale(b["gate"], 0.03)
        be.silu_mul(b["gate"], b["up"])
        be.matmul(ih.weights(wd, ih.NVFP4, 256, nd), b["h"], b["out"])
        be.scale(b["out"], 0.5)
    run(pair, n, b, script, ["gate", "out"], at_most=5)


@pytest.mark.parametrize("n,nd,ff,scaled", [(40, 512, 64, True), (131, 768, 68, False), (200, 1024, 128, True), (1030, 512, 96, True)])
def test_the_nvfp4_shared_experts_up_product_stays_readable(pair, n, nd, ff, scaled):
    """The gate and up products in one launch leave the up product where an op or the host finds it: behind the gated product
    (with the row lengths of either 16-wide kernel and of the 128-wide one)."""
    import inferred_hip as ih
    r = rng(8)
    wg, wu, wd = nvfp4_weights(r, ff, nd), nvfp4_weights(r, ff, nd), q8_0_weights_of(r, 64, 64)
    z = lambda k: np.zeros(k, np.float32)  # noqa: E731
    b = dict(x=f32(r, n * nd, 0.2), gate=z(n * ff), up=z(n * ff), rows=z(n * ff), h=f32(r, n * 64), out=z(n * 64))

    def script(be, b):
        be.matmul(ih.weights(wg, ih.NVFP4, nd, ff), b["x"], b["gate"])
        be.matmul(ih.weights(wu, ih.NVFP4, nd, ff), b["x"], b["up"])
        if scaled:
            be.scale(b["up"], 0.25)
            be.scale(b["gate"], 0.03)
        be.silu_mul(b["gate"], b["up"])
        be.matmul(ih.weights(wd, ih.Q8_0, 64, 64), b["h"], b["out"])
        be.gather_chunks(b["up"], ff, ff, 0, b["rows"])
    run(pair, n, b, script, ["gate", "up", "rows"], at_most=6, other_first=True)
