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
