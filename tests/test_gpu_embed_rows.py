"""The embedding rows made on the device (it_hip_embed_rows) against the host's dequantization, and the single-token passes
that are fed by them in turn with arg-max fed ones (each kind replays a graph of its own)."""
import numpy as np
import pytest

import inferred_hip as ih

pytestmark = pytest.mark.gpu


def table(ty, n_vocab, n_in, r):
    v = r.standard_normal((n_vocab, n_in)).astype(np.float32)
    if ty == ih.F32:
        return v, v
    if ty == ih.F16:
        h = v.astype(np.float16)
        return h, h.astype(np.float32)
    if ty == ih.BF16:
        u = (v.view(np.uint32) >> 16).astype(np.uint16)
        return u, (u.astype(np.uint32) << 16).view(np.float32)
    q = r.integers(-127, 128, (n_vocab, n_in // 32, 32)).astype(np.int8)
    d = (r.random((n_vocab, n_in // 32)) * 0.01).astype(np.float16)
    blk = np.zeros((n_vocab, n_in // 32, 34), np.uint8)
    blk[..., :2] = d.view(np.uint8).reshape(n_vocab, n_in // 32, 2)
    blk[..., 2:] = q.view(np.uint8)
    return blk, (d.astype(np.float32)[..., None] * q.astype(np.float32)).reshape(n_vocab, n_in)


@pytest.mark.parametrize("ty,n_in", [(ih.Q8_0, 32), (ih.Q8_0, 2048), (ih.Q8_0, 2080), (ih.F16, 100), (ih.BF16, 2049), (ih.F32, 7)])
def test_rows_equal_the_host_form(ty, n_in):
    r = np.random.default_rng(n_in)
    raw, want = table(ty, 97, n_in, r)
    be = ih.Hip()
    try:
        w = ih.weights(raw, ty, n_in, 97)
        for n in (1, 2, 300):
            ids = r.integers(0, 97, n).astype(np.uint32)
            ids[-1] = 96
            x = np.zeros(n * n_in, np.float32)
            be.begin_pass(n)
            assert be.L.it_hip_embed_rows(be.h, ih.C.addressof(w), ids.ctypes.data, n, x.ctypes.data, x.size) == 1
            be.end_pass()
            be.host_needs(x)
            assert np.array_equal(x.reshape(n, n_in), want[ids])
            be.release(x)
        ids[0] = 97   # outside the table
        assert be.L.it_hip_embed_rows(be.h, ih.C.addressof(w), ids.ctypes.data, n, x.ctypes.data, x.size) == 0
        be.raise_if_error()
    finally:
        be.close()


def test_passes_of_two_kinds_in_turn_keep_their_graphs(tiny_gguf):
    """generate() takes its prompt's token from the host and feeds the rest on the device; forward() feeds every token."""
    be = ih.Hip(exact=True)
    m = ih.Model(tiny_gguf)
    eng = ih.Engine(m, be, 64, 16)
    try:
        want = None
        for _ in range(4):
            eng.reset()
            ids, last = eng.generate(np.array([7], np.uint32), 12)
            eng.reset()
            fed = [eng.forward(np.array([t], np.uint32)) for t in [7, *ids[:-1]]]
            assert [int(np.argmax(l)) for l in fed] == ids.tolist()
            assert np.array_equal(fed[-1], last)
            want = ids if want is None else want
            assert np.array_equal(ids, want)
        g = be.graph_stats()
        # (one recording may be given up: the attention scratch grows to its graphed size)
        assert g["captures"] == 2 and g["aborts"] <= 1, g
        be.raise_if_error()
    finally:
        eng.close(); m.close(); be.close()


ROWS = {   # what a single-token pass makes of rows of the table: the ops, and the result from the rows
    "two_rows": (lambda be, e, b: (e(b["x"], 0), e(b["y"], 1), be.add_assign(b["x"], b["y"])), lambda r, v: r[0] + r[1]),
    "one_after_the_other": (lambda be, e, b: (e(b["y"], 0), be.add_assign(b["x"], b["y"]), e(b["y"], 1), be.add_assign(b["x"], b["y"])),
                            lambda r, v: (v + r[0]) + r[1]),
    "behind_the_buffers_last_values": (lambda be, e, b: (be.scale(b["x"], 2.0), e(b["x"], 0), be.scale(b["x"], 4.0)), lambda r, v: 4 * r[0]),
    "newer_host_values": (lambda be, e, b: (e(b["x"], 0), b["x"].__setitem__(slice(None), b["v"]), be.host_wrote(b["x"]), be.scale(b["x"], 4.0)),
                          lambda r, v: 4 * v),
}


@pytest.mark.parametrize("what", sorted(ROWS))
def test_rows_in_the_order_of_the_passes_ops(what):
    """A recorded pass makes its one embedding row in front of its ops; a second row, and one whose buffer other ops or the
    host have to do with, keep their place."""
    r = np.random.default_rng(1)
    raw, rows = table(ih.Q8_0, 50, 64, r)
    w = ih.weights(raw, ih.Q8_0, 64, 50)
    be = ih.Hip()
    ops, want = ROWS[what]
    try:
        b = dict(x=np.zeros(64, np.float32), y=np.zeros(64, np.float32), v=np.zeros(64, np.float32))
        for i in range(6):    # op by op, recorded, replayed
            ids = r.integers(0, 50, 2).astype(np.uint32)
            v = r.standard_normal(64).astype(np.float32)
            b["x"][:] = v
            b["v"][:] = v + 1
            be.begin_pass(1)
            be.host_wrote(b["x"])

            def embed(x, k):
                one = ids[k:k + 1].copy()
                assert be.L.it_hip_embed_rows(be.h, ih.C.addressof(w), one.ctypes.data, 1, x.ctypes.data, x.size) == 1
            ops(be, embed, b)
            be.end_pass()
            be.host_needs(b["x"])
            be.raise_if_error()
            at = v + 1 if what == "newer_host_values" else v
            assert np.array_equal(b["x"], want(rows[ids], at).astype(np.float32)), (what, i)
    finally:
        be.close()
