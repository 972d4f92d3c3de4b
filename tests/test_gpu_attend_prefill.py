"""The one-pass prefill attention at its own edges: one, two and three key tiles (its loop handles tiles in pairs), a ragged
last tile, and batches of few blocks, whose keys are cut into shares (more shares than a block has tiles among them)."""
import numpy as np
import pytest
from util import bf16_round, close, f16_bits, rng

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


@pytest.mark.parametrize("n_q,n_pos,hd,nh,nkv", [(64, 64, 256, 4, 4), (65, 65, 128, 4, 2), (128, 128, 64, 2, 2), (129, 129, 256, 16, 1),
                                                 (17, 255, 128, 8, 1), (17, 256, 256, 16, 2), (17, 513, 64, 8, 2), (100, 4097, 256, 16, 2),
                                                 (512, 1700, 256, 16, 2), (33, 9000, 128, 16, 1), (1100, 1100, 64, 1, 1),
                                                 (700, 1000, 128, 2, 2)])
def test_prefill_attention(hip, orc, n_q, n_pos, hd, nh, nkv):
    hip.drop_mirrors(); hip.begin_pass(n_q)
    r = rng(n_pos)
    kv_dim = nkv * hd
    q = bf16_round((3 * r.standard_normal(n_q * nh * hd)).astype(np.float32))   # (peaked rows: the maximum moves from tile to tile)
    k = f16_bits(r.standard_normal(n_pos * kv_dim)); v = f16_bits(r.standard_normal(n_pos * kv_dim))
    a, b = np.zeros(n_q * nh * hd, np.float32), np.zeros(n_q * nh * hd, np.float32)
    sc = 1.0 / np.sqrt(np.float32(hd))
    hip.attend(q, k, v, kv_dim, n_pos, hd, nh, nkv, sc, a); hip.host_needs(a)
    orc.attend(q, k, v, kv_dim, n_pos, hd, nh, nkv, sc, b)
    hip.raise_if_error()
    assert close(a, b), np.abs(a - b).max()
