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
