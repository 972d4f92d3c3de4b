"""it_hip_replay_pass through the C ABI: a tagged single-token pass launched from what earlier ones recorded, up to the last
row of its cache slab and not past it.  The pass (embedding row, rotation, cache write, attention over the context) is also
issued op by op on a backend that records nothing; slabs and outputs are compared bit for bit but for the attention, whose
splits are added in another order there."""
import ctypes as C

import numpy as np
import pytest

from util import assert_bits_equal, close, q8_0_weights, rng

pytestmark = pytest.mark.gpu
HD, NH, VOCAB = 64, 2, 40
DIM = HD * NH


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("rows", [12, 70])
def test_replayed_up_to_the_end_of_the_slab(rows, exact):
    import inferred_hip as ih
    from oracle import binding as ob
    r = rng(3)
    table = q8_0_weights(ob.Oracle(threads=2), r, VOCAB, DIM, std=1.0)
    tw = ih.weights(table, ih.Q8_0, DIM, VOCAB)
    ids = r.integers(0, VOCAB, rows + 2).astype(np.uint32)
    tag = np.zeros(1, np.uint8)
    backends = [ih.Hip(exact=exact), ih.Hip(exact=exact, graph=False)]
    try:
        states = []
        for be in backends:
            x, out = np.zeros(DIM, np.float32), np.zeros(DIM, np.float32)
            # the slab ends where the page does not: a row past it would be another tensor's
            k, v = (np.zeros(rows * DIM, np.uint16) for _ in range(2))
            states.append((be, x, out, k, v))

        def issue(be, x, out, k, v, pos):
            one = ids[pos:pos + 1].copy()
            be.begin_pass(1)
            be.L.it_hip_tag_pass(be.h, tag.ctypes.data, pos)
            assert be.L.it_hip_embed_rows(be.h, C.addressof(tw), one.ctypes.data, 1, x.ctypes.data, x.size)
            be.rope_neox(x, pos, HD, HD, NH, 1e4)
            be.kv_write(k, pos * DIM, x)
            be.kv_write(v, pos * DIM, x)
            be.attend(x, k, v, DIM, pos + 1, HD, NH, NH, 0.125, out)
            be.end_pass()

        replayed = 0
        for pos in range(rows):
            got = []
            for be, x, out, k, v in states:
                one = ids[pos:pos + 1].copy()
                if be.L.it_hip_replay_pass(be.h, tag.ctypes.data, pos, one.ctypes.data, 0):
                    assert be is backends[0]
                    replayed += 1
                else:
                    issue(be, x, out, k, v, pos)
                be.host_needs(out)
                be.raise_if_error()
                got.append(out.copy())
            assert close(got[0], got[1], 1e-5), pos
        assert replayed >= rows // 4, replayed
        be, x, out, k, v = states[0]
        one = ids[rows:rows + 1].copy()
        for pos in (rows, rows + 1, 1 << 20, (1 << 31) - 1, 1 << 31, 1 << 40, (1 << 64) - 1):
            assert be.L.it_hip_replay_pass(be.h, tag.ctypes.data, pos, one.ctypes.data, 0) == 0, pos
        issue(be, x, out, k, v, rows)     # what the caller does then: the op refuses the row
        err = be.take_error()
        assert err is not None and "kv_write" in err, err
        for be, *_, k, v in states:
            be.read_kv(k)
            be.read_kv(v)
            assert be.take_error() is None
        for a, b in zip(states[0][3:], states[1][3:]):
            assert_bits_equal(a.view(np.float16).astype(np.float32), b.view(np.float16).astype(np.float32), "cache")
            assert (a.reshape(rows, DIM)[-1] != 0).any()
    finally:
        for be in backends:
            be.take_error()
            be.close()


@pytest.mark.parametrize("host_values", [False, True])
def test_a_pass_that_takes_values_from_the_host_is_issued_every_time(host_values):
    """x = a row of the table, then x += a vector: of the device (made by the pass before) or of the host (new in each pass)."""
    import inferred_hip as ih
    from oracle import binding as ob
    r = rng(4)
    orc = ob.Oracle(threads=2)
    raw = q8_0_weights(orc, r, VOCAB, DIM, std=1.0)
    tw = ih.weights(raw, ih.Q8_0, DIM, VOCAB)
    blocks = raw.reshape(VOCAB, DIM // 32, 34)
    rows = (blocks[..., :2].copy().view(np.float16).astype(np.float32) * blocks[..., 2:].view(np.int8).astype(np.float32)).reshape(VOCAB, DIM)
    tag = np.zeros(1, np.uint8)
    be = ih.Hip()
    try:
        x, v = np.zeros(DIM, np.float32), np.zeros(DIM, np.float32)
        replayed = 0
        for pos in range(10):
            one = r.integers(0, VOCAB, 1).astype(np.uint32)
            v[:] = r.standard_normal(DIM)
            if be.L.it_hip_replay_pass(be.h, tag.ctypes.data, pos, one.ctypes.data, 0):
                replayed += 1
            else:
                be.begin_pass(1)
                be.L.it_hip_tag_pass(be.h, tag.ctypes.data, pos)
                assert be.L.it_hip_embed_rows(be.h, C.addressof(tw), one.ctypes.data, 1, x.ctypes.data, x.size)
                if host_values:
                    be.host_wrote(v)
                    be.add_assign(x, v)
                else:
                    be.add_assign(x, x)
                be.end_pass()
            be.host_needs(x)
            be.raise_if_error()
            assert np.array_equal(x, rows[one[0]] + (v if host_values else rows[one[0]])), pos
        assert replayed == 0 if host_values else replayed >= 4, replayed
    finally:
        be.close()
