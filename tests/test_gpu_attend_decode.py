"""The few-query attention over caches that hold infinities and NaN: a query's row depends on the keys and values up to its
own position, whatever stands in the rows behind it (two queries of a verify batch share a block, and the later one's key lies
in the earlier one's tile)."""
import numpy as np
import pytest

from util import close, f16_bits, rng

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import inferred_hip as ih
    be = ih.Hip(exact=False)
    yield be
    err = be.take_error()
    be.close()
    assert err is None, err


@pytest.fixture(scope="module")
def orc():
    from oracle import binding as ob
    return ob.Oracle(threads=8)


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("hd,nh,nkv", [(64, 8, 2), (128, 8, 1), (256, 16, 2), (256, 4, 4)])
# the later key first, last and in the middle of a tile and of its range; pairs and a query left over
@pytest.mark.parametrize("n_q,n_pos", [(2, 2), (2, 64), (2, 65), (3, 66), (4, 200), (5, 1039), (8, 17000)])
def test_a_row_does_not_depend_on_what_stands_behind_it(hip, orc, n_q, n_pos, hd, nh, nkv, bad):
    r = rng(n_pos + hd)
    kv_dim = nkv * hd
    q = r.standard_normal(n_q * nh * hd).astype(np.float32)
    k = r.standard_normal((n_pos, kv_dim)).astype(np.float16)
    v = r.standard_normal((n_pos, kv_dim)).astype(np.float16)
    sc = 1.0 / np.sqrt(np.float32(hd))

    def attend(be, k, v):
        out = np.zeros(n_q * nh * hd, np.float32)
        if be is hip:
            hip.drop_mirrors(); hip.begin_pass(n_q)
        be.attend(q, f16_bits(k).reshape(-1), f16_bits(v).reshape(-1), kv_dim, n_pos, hd, nh, nkv, sc, out)
        if be is hip:
            hip.host_needs(out); hip.end_pass(); hip.raise_if_error()
        return out.reshape(n_q, nh, hd)
    want = attend(orc, k, v)
    assert close(attend(hip, k, v), want)
    for t in sorted({0, n_q - 2}):        # the rows behind query t's position, all of them bad in one dim of every head
        kb, vb = k.copy(), v.copy()
        behind = n_pos - n_q + 1 + t
        kb[behind:, 1::hd] = bad
        vb[behind:, 3::hd] = bad
        got = attend(hip, kb, vb)
        assert close(got[:t + 1], want[:t + 1]), (t, np.abs(got[:t + 1] - want[:t + 1]).max())
        assert not np.isfinite(got[t + 1:, :, 3]).any()


@pytest.mark.parametrize("hd,nh,nkv", [(64, 8, 2), (128, 8, 1), (256, 4, 4)])
@pytest.mark.parametrize("n_pos", [9, 40, 70, 71, 1039])
def test_an_infinite_value_counts_with_its_own_keys_weight(hip, orc, n_pos, hd, nh, nkv):
    # two queries; the last key, which only the second sees, holds an infinity.  Scores of 0 and, in turn, of the last key or of
    # all the others 200 lower, a weight of zero in f32 too: 0 x inf is not a number, any other weight's product an infinity
    r = rng(n_pos + hd)
    kv_dim = nkv * hd
    q = np.zeros((2, nh, hd), np.float32)
    q[..., 0] = 1.0
    v = r.standard_normal((n_pos, kv_dim)).astype(np.float16)
    v[-1, 3::hd] = np.inf
    for last, others in ((0.0, 0.0), (0.0, -200.0), (-200.0, 0.0)):
        k = np.zeros((n_pos, kv_dim), np.float16)
        k[:, ::hd] = others
        k[-1, ::hd] = last
        rows = []
        for be in (hip, orc):
            out = np.zeros(q.size, np.float32)
            if be is hip:
                hip.drop_mirrors(); hip.begin_pass(2)
            be.attend(q.reshape(-1), f16_bits(k).reshape(-1), f16_bits(v).reshape(-1), kv_dim, n_pos, hd, nh, nkv, np.float32(1.0), out)
            if be is hip:
                hip.host_needs(out); hip.end_pass(); hip.raise_if_error()
            rows.append(out.reshape(2, nh, hd))
        got, want = rows
        assert np.isfinite(want[0]).all() and np.isfinite(got[0]).all(), (last, others)
        assert np.array_equal(np.isnan(got[1]), np.isnan(want[1])), (last, others)
        assert np.array_equal(np.isposinf(got[1]), np.isposinf(want[1])), (last, others)
        assert close(np.nan_to_num(got, posinf=0), np.nan_to_num(want, posinf=0))


@pytest.mark.parametrize("hd,nh,nkv", [(64, 8, 2), (128, 8, 1), (256, 4, 4)])
# eight queries, whose seven later keys stand in one slice of 32 keys or on both sides of an edge, in one range and in several
@pytest.mark.parametrize("n_pos", [35, 38, 40, 67, 131, 1031])
def test_infinite_values_of_later_keys_count_with_their_last_weight(hip, orc, n_pos, hd, nh, nkv):
    # One of the keys that only later queries see holds infinities, and scores 40 or 200 below or above a key before or behind it: a
    # weight of 4e-18 is one in f32 (and no f16), one of 1e-87 is not.  A key behind it raises the maximum after it was seen.
    r = rng(n_pos * 7 + hd)
    n_q, kv_dim = 8, nkv * hd
    q = np.zeros((n_q, nh, hd), np.float32)
    q[..., 0] = 1.0
    values = r.standard_normal((n_pos, kv_dim)).astype(np.float16)
    first = n_pos - n_q + 1                                    # the first key that not every query sees
    for bad in range(first, n_pos):
        for high in sorted({first, bad - 1, bad, n_pos - 1}):      # the key whose score is above all others'
            for gap in (40.0, 200.0):
                k, v = np.full((n_pos, kv_dim), 0, np.float16), values.copy()
                k[high, ::hd] = gap
                v[bad, 3::hd], v[bad, 5::hd] = np.inf, -np.inf
                rows = []
                for be in (hip, orc):
                    out = np.zeros(q.size, np.float32)
                    if be is hip:
                        hip.drop_mirrors(); hip.begin_pass(n_q)
                    be.attend(q.reshape(-1), f16_bits(k).reshape(-1), f16_bits(v).reshape(-1), kv_dim, n_pos, hd, nh, nkv, np.float32(1.0), out)
                    if be is hip:
                        hip.host_needs(out); hip.end_pass(); hip.raise_if_error()
                    rows.append(out.reshape(n_q, nh, hd))
                got, want = rows
                for kind in (np.isnan, np.isposinf, np.isneginf):
                    assert np.array_equal(kind(got), kind(want)), (kind.__name__, bad - first, high - first, gap)
                assert close(np.nan_to_num(got, posinf=0, neginf=0), np.nan_to_num(want, posinf=0, neginf=0)), (bad - first, high - first, gap)


@pytest.mark.parametrize("hd,nh,nkv", [(64, 8, 2), (64, 4, 4), (128, 8, 1), (128, 32, 4), (256, 16, 2), (256, 4, 2)])
# one query to two groups of eight; contexts around a wave's quarter (8), a slice (32), a stage (64, 128) and a round of ranges
@pytest.mark.parametrize("n_q", [1, 2, 3, 4, 5, 8, 9, 16])
def test_queries_and_contexts_around_the_tiles_edges(hip, orc, n_q, hd, nh, nkv):
    sc = 1.0 / np.sqrt(np.float32(hd))
    for n_pos in (n_q, 31, 32, 33, 64, 65, 127, 128, 129, 257, 1000, 8193, 16400):
        if n_pos < n_q:
            continue
        r = rng(n_pos * 31 + n_q)
        kv_dim = nkv * hd
        q = r.standard_normal(n_q * nh * hd).astype(np.float32)
        k, v = f16_bits(r.standard_normal(n_pos * kv_dim)), f16_bits(r.standard_normal(n_pos * kv_dim))
        out, want = np.zeros(n_q * nh * hd, np.float32), np.zeros(n_q * nh * hd, np.float32)
        orc.attend(q, k, v, kv_dim, n_pos, hd, nh, nkv, sc, want)
        hip.drop_mirrors(); hip.begin_pass(n_q)
        hip.attend(q, k, v, kv_dim, n_pos, hd, nh, nkv, sc, out)
        hip.host_needs(out); hip.end_pass(); hip.raise_if_error()
        # probabilities are f16: 2^-11 of the largest value a row's average can hold
        assert np.abs(out - want).max() <= 1e-3, (n_q, n_pos, np.abs(out - want).max())


@pytest.mark.parametrize("n_q,n_pos", [(1, 5), (1, 700), (2, 700), (4, 333), (7, 1500)])
def test_operands_that_are_not_16_byte_aligned(n_q, n_pos):
    import inferred_hip as ih
    from util import Hiprt
    hd, nh, nkv = 128, 16, 4
    r = rng(n_pos)
    kv = n_pos * nkv * hd
    q = r.standard_normal(n_q * nh * hd).astype(np.float32)
    k, v = f16_bits(r.standard_normal(kv)), f16_bits(r.standard_normal(kv))
    rt = Hiprt()
    try:
        got = []
        for shift in (0, 1):   # q one float further, K and V one half further
            dq = rt.upload(np.concatenate([np.zeros(shift, np.float32), q]))
            dk, dv = (rt.upload(np.concatenate([np.zeros(shift, np.uint16), x])) for x in (k, v))
            dout = rt.filled(q.nbytes, 0xff)
            rc, msg = ih.attend_noalloc(dq + 4 * shift, q.size, dk + 2 * shift, dv + 2 * shift, kv, nkv * hd, n_pos, hd, nh, nkv,
                                        float(hd ** -0.5), dout, q.size, stream=0)
            assert rc == 0, msg
            got.append(rt.download(dout, np.zeros_like(q)))
        assert np.isfinite(got[0]).all()
        assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
    finally:
        rt.free_all()
